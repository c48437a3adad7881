"""GPU: the 32-points-per-thread column kernel (512 to 4096 points) in each of
its workgroup sizes, on matrices narrower than a group, groups that span
batch items, partial last groups, and rows that do not start on 128-byte
lines (by their length or by the buffer's address), against the FP64 oracle.

Tolerance: a length-n FP32 transform rounds about log2(n) <= 12 times per
value, 6e-8 each, and its twiddles once or twice more: relative L2 per column
<= 1e-6."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6

# (n, ncols, batch): few columns (256 threads, and the split passes of 4096),
# from 256 groups of 16384 points on 512 threads, of 32768 points 1024
SHAPES = [(512, 1, 5), (512, 33, 3), (512, 31, 300), (512, 64, 200), (1024, 15, 3), (1024, 17, 250), (1024, 48, 100),
          (1024, 64, 130), (2048, 3, 5), (2048, 30, 40), (2048, 7, 320), (2048, 16, 257), (4096, 1, 3),
          (4096, 11, 100), (4096, 9, 230), (4096, 16, 129),
          # between one 256-, 512- and 1024-thread workgroup per CU, and the two-pass split's ragged rows
          (1024, 256, 10), (1024, 256, 21), (2048, 256, 9), (4096, 64, 17), (512, 256, 50), (1024, 333, 17),
          (4096, 20, 50),
          # shorter columns (16 points per thread): windows, and 16 points on both sides of 2^23
          (16, 167, 50), (16, 999, 530), (32, 100, 90), (128, 2048, 17), (256, 64, 300)]


def _columns(x, sign):
    import torch
    from bfly import ops
    y = ops.fft_columns(x, sign)
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("offset", [0, 3], ids=["line", "offset3"])
@pytest.mark.parametrize("n,ncols,batch", SHAPES, ids=[f"{a}x{b}x{c}" for a, b, c in SHAPES])
def test_wide_columns_against_the_oracle(n, ncols, batch, offset):
    import torch
    sign = -1 if batch % 2 else 1
    print(f"columns n={n} ncols={ncols} batch={batch} sign={sign} offset={offset}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + ncols + batch)
    flat = torch.rand(offset + n * ncols * batch, 2, generator=g, device="cuda") * 2 - 1
    x = torch.view_as_complex(flat)[offset:].view(batch, n, ncols)
    y = _columns(x, sign)
    total = ncols * batch
    # the ends, every column around a group boundary of the first groups, a spread
    pick = sorted({c for c in [*range(34), *range(total - 34, total), *range(0, total, max(1, total // 40))]
                   if 0 <= c < total})
    b, c = np.array(pick) // ncols, np.array(pick) % ncols

    def rows(t):
        return torch.view_as_real(t[b, :, c]).cpu().numpy().reshape(len(pick), 2 * n)

    assert oracle.rel_l2_rows(rows(y), oracle.c2c_f64(rows(x), n, sign)) <= REL_L2


@pytest.mark.parametrize("n,ncols,batch", [(1024, 64, 130), (2048, 16, 257)])
def test_wide_columns_do_not_depend_on_the_workgroup(n, ncols, batch):
    # one call (1024 threads) equals calls on slices of the batch (512 and
    # 256 threads) bit for bit: the per-column arithmetic is the same
    import torch
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.view_as_complex(torch.rand(batch, n, ncols, 2, generator=g, device="cuda") * 2 - 1)
    y = _columns(x, -1)
    half, few = batch // 2 + 1, 3
    assert torch.equal(y[:half], _columns(x[:half], -1))
    assert torch.equal(y[:few], _columns(x[:few], -1))
