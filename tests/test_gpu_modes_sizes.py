"""GPU: C2R of spectra truncated to between two and four sixteenths, on both
sides of the batch sizes where the pruned kernel takes over from the full one
and back: bit for bit the transform of the spectrum padded with zeros."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch,bins", [
    (4096, 1536, 512), (4096, 1537, 512), (4096, 4096, 300), (4096, 4097, 300), (2048, 6144, 256), (2048, 6145, 129),
    (1024, 8192, 128), (1024, 8193, 128), (512, 12289, 33), (512, 28671, 64), (512, 28672, 47), (512, 28672, 48)])
def test_truncated_c2r_equals_the_padded_one(n, batch, bins):
    import torch
    from bfly import _lib, ops
    lib, s = _lib.hip(), torch.cuda.current_stream().cuda_stream
    print(f"c2r n={n} batch={batch} bins={bins}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + batch + bins)
    h = torch.rand(batch, 2 * bins, generator=g, device="cuda") * 2 - 1
    padded = torch.zeros(batch, n + 2, device="cuda")
    padded[:, :2 * bins] = h
    y, want = (torch.full((batch, n), float("nan"), device="cuda") for _ in range(2))
    tab = ops.table(_lib.KIND_C2R, n, h.device).data_ptr()
    for src, dst, k in ((h, y, bins), (padded, want, n // 2 + 1)):
        assert lib.bfly_real_ex(_lib.KIND_C2R, src.data_ptr(), dst.data_ptr(), n, batch, k, 2 * k,
                                _lib.VARIANT_STREAM_LT, 0, tab, s) == 0
    torch.cuda.synchronize()
    assert torch.equal(y, want)
