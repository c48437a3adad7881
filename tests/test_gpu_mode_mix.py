"""GPU: bfly_mode_mix at the sizes where its tiles, chunks and mode groups end
(one row / column / mode beyond or short of a tile, odd and single modes,
every tile shape), on operands that start 8 bytes off a 16-byte boundary and
carry NaN around them.

Tolerance: sums of at most 132 products of normal numbers in FP32, relative
to the largest result: 6e-8 * sqrt(2 * 132) < 1e-6."""
import pytest

pytestmark = pytest.mark.gpu

# (batch, c_in, c_out, modes): 16 x 16 tiles, 16 x 32 and 32 x 32 ones
SIZES = [(1, 1, 1, 1), (2, 9, 3, 1), (1, 8, 16, 2), (16, 16, 16, 8), (17, 7, 17, 9), (15, 33, 31, 7),
         (16, 24, 128, 513), (5, 132, 100, 255), (64, 16, 130, 257), (65, 130, 127, 250)]


def _operand(torch, g, shape):
    """A complex64 tensor inside a buffer of NaN, 8 bytes past a 16-byte boundary."""
    n = 1
    for s in shape:
        n *= s
    buf = torch.full((n + 6, 2), float("nan"), device="cuda")
    buf[3:3 + n] = torch.randn(n, 2, generator=g, device="cuda")
    return torch.view_as_complex(buf)[3:3 + n].view(shape)


@pytest.mark.parametrize("B,ci,co,K", SIZES, ids=["x".join(map(str, s)) for s in SIZES])
def test_mode_mix_edges(B, ci, co, K):
    import torch
    from bfly import _lib
    lib = _lib.hip()
    g = torch.Generator(device="cuda").manual_seed(B * 7 + K)
    x, w, gy = _operand(torch, g, (B, ci, K)), _operand(torch, g, (ci, co, K)), _operand(torch, g, (B, co, K))
    x64, w64, gy64 = (t.cpu().to(torch.complex128).permute(2, 0, 1).contiguous() for t in (x, w, gy))
    want = {_lib.MIX_FORWARD: (x, w, torch.bmm(x64, w64)),
            _lib.MIX_GRAD_INPUT: (gy, w, torch.bmm(gy64, w64.conj().transpose(1, 2).contiguous())),
            _lib.MIX_GRAD_WEIGHT: (x, gy, torch.bmm(x64.conj().transpose(1, 2).contiguous(), gy64))}
    for op, (a, b, ref) in want.items():
        print(f"mode_mix op={op} B={B} ci={ci} co={co} K={K}", flush=True)
        ref = ref.permute(1, 2, 0)
        out = torch.full((ref.numel() + 6,), complex(7, -7), dtype=torch.complex64, device="cuda")
        rc = lib.bfly_mode_mix(op, a.data_ptr(), b.data_ptr(), out[3:].data_ptr(), B, ci, co, K,
                               torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        torch.cuda.synchronize()
        got = out[3:-3].cpu().to(torch.complex128).view(ref.shape)
        assert ((got - ref).abs().max() / ref.abs().max()).item() < 1e-6, op
        assert bool((out[:3] == complex(7, -7)).all()) and bool((out[-3:] == complex(7, -7)).all())
