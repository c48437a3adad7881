"""GPU: mode-truncated R2C and C2R (bfly_real_ex, LDS-twiddle streaming form)
around the bin counts where their pruned kernels begin and end, on ragged and
multi-round batches, forward and adjoint.

The pruned kernels leave out only arithmetic on values that are zero or not
stored, so they equal the full-spectrum kernels of the same form bit for bit
(which the parity tests hold to FP64): R2C the first bins of the full
spectrum, C2R the transform of the spectrum padded with zeros.  Rows lie
further apart than their bins, and the gaps stay untouched."""
import pytest

pytestmark = pytest.mark.gpu

LAST = {128: 8, 256: 16, 512: 2, 1024: 4, 2048: 8, 4096: 16}  # radix of the n/2-point plan's last pass


def _cases():
    for m, last in LAST.items():
        edges = {1, m // 8 - 1, m // 8, m // 8 + 1, m // 4, m // 4 + 1, m // last, m // last + 1}
        for bins in sorted(edges):
            yield 2 * m, bins


@pytest.mark.parametrize("n,bins", list(_cases()))
def test_truncated_equals_full_bit_for_bit(n, bins):
    import torch
    from bfly import _lib, ops
    lib, s = _lib.hip(), torch.cuda.current_stream().cuda_stream
    stride, whole = 2 * bins + 6, n + 2

    def run(kind, src, dst, b, k, ld, adj):
        assert lib.bfly_real_ex(kind, src.data_ptr(), dst.data_ptr(), n, b, k, ld, _lib.VARIANT_STREAM_LT, adj,
                                ops.table(kind, n, src.device).data_ptr(), s) == 0

    # one row, a ragged unit, several units per resident workgroup
    for b in (1, 37, (1 << 24) // n + 3):
        print(f"modes n={n} bins={bins} b={b}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(n + bins)
        x = torch.rand(b, n, generator=g, device="cuda") * 2 - 1
        h = torch.rand(b, stride, generator=g, device="cuda") * 2 - 1
        padded = torch.zeros(b, whole, device="cuda")
        padded[:, :2 * bins] = h[:, :2 * bins]
        for adj in (0, _lib.REAL_ADJOINT):
            y, full = torch.full((b, stride), 7.0, device="cuda"), torch.empty(b, whole, device="cuda")
            run(1, x, y, b, bins, stride, adj)
            run(1, x, full, b, n // 2 + 1, whole, adj)
            z, want = (torch.full((b, n), float("nan"), device="cuda") for _ in range(2))
            run(2, h, z, b, bins, stride, adj)
            run(2, padded, want, b, n // 2 + 1, whole, adj)
            torch.cuda.synchronize()
            assert torch.equal(y[:, :2 * bins], full[:, :2 * bins]), ("r2c", b, adj)
            assert bool((y[:, 2 * bins:] == 7.0).all())
            assert torch.equal(z, want), ("c2r", b, adj)
