"""GPU: the entry points that share AUTO's kernels agree with bfly_c2c bit for
bit on both sides of each size where AUTO changes kernel (the allocation-free
call, contiguous rows), and column results that different kernels compute for
other batches or alignments agree to their rounding."""
import pytest

pytestmark = pytest.mark.gpu


def _uniform(seed, *shape):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(*shape, generator=g, device="cuda") * 2 - 1


@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("n,b", [(8192, 127), (8192, 128), (16384, 159), (16384, 160), (16384, 256), (32768, 128),
                                 (32768, 129), (32768, 256)])
def test_noalloc_and_rows_equal_bfly_c2c(n, b, sign):
    import torch
    from bfly import _lib, ops
    lib, s = _lib.hip(), torch.cuda.current_stream().cuda_stream
    print(f"routes n={n} b={b} sign={sign}", flush=True)
    x = _uniform(n + b, b, 2 * n)
    held = torch.empty_like(x)
    tab, work = ops.table(_lib.KIND_C2C, n, x.device).data_ptr(), held.data_ptr()
    want, got, rows = (torch.full_like(x, float("nan")) for _ in range(3))
    assert lib.bfly_c2c(x.data_ptr(), want.data_ptr(), n, b, sign, tab, work, s) == 0
    assert lib.bfly_c2c_noalloc(x.data_ptr(), got.data_ptr(), n, b, sign, tab, s) == 0
    assert lib.bfly_c2c_rows(x.data_ptr(), n, rows.data_ptr(), n, n, b, sign, tab, work, s) == 0
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    if n == 32768:
        assert torch.equal(rows, want)
    else:  # the LDS-twiddle streaming form
        lt = torch.full_like(x, float("nan"))
        assert lib.bfly_c2c_ex(x.data_ptr(), lt.data_ptr(), n, b, sign, _lib.VARIANT_STREAM_LT, tab, work, s) == 0
        torch.cuda.synchronize()
        assert torch.equal(rows, lt)


@pytest.mark.parametrize("n,ncols,batch,part", [(512, 64, 200, 100), (1024, 64, 130, 40), (4096, 64, 17, 3),
                                                (2048, 16, 257, 5), (1024, 12, 400, 20)])
def test_columns_of_another_batch_or_alignment(n, ncols, batch, part):
    import torch
    from bfly import ops
    print(f"columns n={n} ncols={ncols} batch={batch} part={part}", flush=True)
    flat = torch.view_as_complex(_uniform(n + ncols, batch * n * ncols + 3, 2))
    x = flat[:-3].view(batch, n, ncols)
    y = ops.fft_columns(x)
    shifted = torch.empty_like(flat)[3:].view(batch, n, ncols)
    shifted.copy_(x)
    # two FP32 transforms, each within 1.4e-7 of the exact one
    for other in (ops.fft_columns(x[:part]), ops.fft_columns(shifted)[:part]):
        assert ((y[:part] - other).norm() / other.norm()).item() <= 2.8e-7
