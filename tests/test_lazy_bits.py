"""Tensors that torch conjugates or negates lazily (a bit of the tensor, the
memory unchanged) through the entry points that take them: the result is that
of the values, not of the memory.  ops.c2c and ops.fft2 refuse lazy conjugates
(test_ops_streams)."""
import pytest
import torch

from bfly import _lib, ops, spectral


def _z(*shape, seed=3, device="cpu"):
    g = torch.Generator().manual_seed(seed)
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g)).to(device)


def test_plain_holds_the_values():
    z = _z(4, 8)
    for t in (z.conj(), torch._neg_view(z), torch._neg_view(z.conj()), z.conj().imag, z):
        p = ops.plain(t)
        assert not p.is_conj() and not p.is_neg()
        assert torch.equal(p, t.clone())
    assert ops.plain(z) is z


@pytest.mark.gpu
def test_columns_and_rows():
    x = _z(3, 64, 20, device="cuda")
    assert torch.equal(ops.fft_columns(x.conj()), ops.fft_columns(x.conj().resolve_conj()))
    assert torch.equal(ops.fft_columns(torch._neg_view(x)), -ops.fft_columns(x))
    pad = _z(5, 70, device="cuda")[:, :64]
    want = ops.c2c_rows(pad.conj().resolve_conj().contiguous())
    assert torch.equal(ops.c2c_rows(pad.conj()), want)
    for out in (torch.empty(5, 64, dtype=torch.complex64, device="cuda").conj(),
                torch._neg_view(torch.empty(5, 64, dtype=torch.complex64, device="cuda"))):
        with pytest.raises(RuntimeError):
            ops.c2c_rows(pad, out=out)


@pytest.mark.gpu
def test_negated_views_of_the_other_transforms():
    x = _z(2, 64, 64, device="cuda")
    r, h = x.real.contiguous(), torch.view_as_real(_z(3, 33, device="cuda")).reshape(3, 66)
    for call, t in ((ops.c2c, x), (ops.fft2, x), (ops.c2c, r), (ops.rfft, r), (lambda v: ops.irfft(v, 64), h),
                    (lambda v: ops.rfft_modes(v, 8), r), (lambda v: ops.irfft_modes(v, 256), r)):
        assert torch.equal(call(torch._neg_view(t)), -call(t))


@pytest.mark.gpu
def test_mode_mix_and_its_gradients():
    B, ci, co, K = 3, 5, 4, 9
    x, w = _z(B, ci, K, device="cuda"), _z(ci, co, K, seed=4, device="cuda")
    whole = lambda t: t.conj().resolve_conj()  # noqa: E731
    got = ops.mode_mix(_lib.MIX_FORWARD, x.conj(), w.conj(), B, ci, co, K)
    assert torch.equal(got, ops.mode_mix(_lib.MIX_FORWARD, whole(x), whole(w), B, ci, co, K))

    def grads(mix):
        a, b = x.clone().requires_grad_(), w.clone().requires_grad_()
        y = mix(a, b.conj()).conj()
        return torch.autograd.grad(y, (a, b), _z(B, co, K, seed=5, device="cuda"))

    def reference(a, b):  # sums of ci, co or B products, in 64 bits on the host
        a, b = a.cpu().to(torch.complex128), b.cpu().to(torch.complex128)
        return (a.permute(2, 0, 1) @ b.resolve_conj().permute(2, 0, 1)).permute(1, 2, 0).to(torch.complex64).cuda()

    # FP32 sums of at most 5 products: 1e-6 of the largest result
    for g, want in zip(grads(spectral.mix_modes), grads(reference)):
        assert ((g - want).abs().max() / want.abs().max()).item() < 1e-6
