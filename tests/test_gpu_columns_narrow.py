"""GPU: column transforms at every form the column kernels launch in -- narrow
matrices alone, in groups of whole matrices and numbered through the batch,
few and many workgroups, every order of tables and loads, each workgroup size
of the 32-point kernel -- on buffers that start on a 128-byte line and off
one, against the FP64 oracle, every column of the first and last matrices and
a spread of the others.

Tolerance: a length-n FP32 transform rounds about log2(n) <= 12 times per
value, 6e-8 each, and its twiddles once or twice more: relative L2 per column
<= 1e-6."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

REL_L2 = 1e-6

# (n, ncols, batch)
SHAPES = [
    # whole groups: up to 512 workgroups, 513 to 1024, beyond
    (64, 256, 75), (64, 64, 700), (64, 64, 1100), (128, 32, 300), (128, 64, 301), (128, 32, 2600), (256, 16, 600),
    (256, 16, 1100), (32, 128, 600), (16, 256, 20), (512, 16, 300), (512, 16, 520),
    # narrow matrices: one or a few to a workgroup, spread over the CUs
    (16, 1, 300), (16, 3, 20), (16, 16, 100), (32, 1, 1500), (32, 5, 60), (64, 1, 120), (64, 7, 100), (128, 1, 20),
    (128, 33, 7), (256, 1, 600), (256, 3, 200), (512, 1, 60), (512, 5, 4), (1024, 1, 30), (1024, 3, 60), (2048, 1, 9),
    # from 2^20 points, with the streaming hint: full, idle lanes, 513 to 1024 workgroups
    (16, 100, 700), (64, 24, 700), (128, 20, 500), (256, 12, 600), (256, 5, 1500), (512, 12, 400), (512, 8, 300),
    # many groups with idle lanes, through the batch
    (16, 100, 600), (64, 40, 400), (256, 3, 1500),
    # 256, 512 and 1024 threads of the 32-point kernel on narrow matrices
    (1024, 12, 50), (1024, 12, 200), (1024, 8, 800), (1024, 7, 300), (2048, 3, 400), (2048, 5, 200), (2048, 12, 150),
    (4096, 3, 350), (4096, 7, 150), (4096, 1, 1100),
    # 2^20 points and more where a wave stores parts of lines; 512-point ones from 4096 columns
    (256, 5, 900), (64, 39, 500), (512, 1, 5000), (512, 7, 600),
    # the 4096-point split: second pass ragged of 16 columns and more in few and many workgroups, and of fewer
    (4096, 20, 8), (4096, 100, 7), (4096, 5, 60), (4096, 5, 3), (4096, 7, 100),
    # 16 points, ragged: spread
    (16, 300, 20), (16, 999, 70)]


@pytest.mark.parametrize("offset", [0, 3], ids=["line", "offset3"])
@pytest.mark.parametrize("n,ncols,batch", SHAPES, ids=[f"{a}x{b}x{c}" for a, b, c in SHAPES])
def test_columns_against_the_oracle(n, ncols, batch, offset):
    import torch
    from bfly import ops
    sign = 1 if ncols % 2 else -1
    print(f"columns n={n} ncols={ncols} batch={batch} sign={sign} offset={offset}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + ncols + batch)
    flat = torch.rand(offset + n * ncols * batch, 2, generator=g, device="cuda") * 2 - 1
    x = torch.view_as_complex(flat)[offset:].view(batch, n, ncols)
    y = ops.fft_columns(x, sign)
    torch.cuda.synchronize()
    total = ncols * batch
    pick = sorted({c for c in [*range(40), *range(total - 40, total), *range(0, total, max(1, total // 60))]
                   if 0 <= c < total})
    b, c = np.array(pick) // ncols, np.array(pick) % ncols

    def rows(t):
        return torch.view_as_real(t[b, :, c]).cpu().numpy().reshape(len(pick), 2 * n)

    assert oracle.rel_l2_rows(rows(y), oracle.c2c_f64(rows(x), n, sign)) <= REL_L2
    # every other column: a second transform the other way gives x n back
    back = ops.fft_columns(y, -sign)
    assert ((back - n * x).abs().max() / n).item() <= 1e-5
