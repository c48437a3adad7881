"""GPU: AUTO's one-transform-per-workgroup kernel of 8192, 16384 and 32768
points (32 points per thread) at the batches around its thresholds, a ragged
multi-round batch, scaled and through padded rows, against the FP64 oracle.

Tolerance: an FP32 transform of 2^15 points rounds about 15 times per value,
6e-8 each, and its twiddles up to three times: relative L2 per transform
<= 2e-6."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

REL_L2 = 2e-6

# below, at and above the batch from which AUTO picks the kernel; more than one
# round of resident workgroups
CASES = [(8192, 127), (8192, 128), (8192, 1301), (16384, 159), (16384, 160), (16384, 255), (16384, 256),
         (16384, 601), (32768, 128), (32768, 129), (32768, 301),
         # the two-kernel chain on both sides of the size from which its intermediate's stores are ordinary ones
         (65536, 64), (65536, 65)]


def _rows(t, pick, n):
    import torch
    return torch.view_as_real(t[pick]).cpu().numpy().reshape(len(pick), 2 * n)


@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("n,b", CASES, ids=[f"{n}x{b}" for n, b in CASES])
def test_auto_long_rows_against_the_oracle(n, b, sign):
    import torch
    from bfly import ops
    print(f"auto n={n} b={b} sign={sign}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + b)
    x = torch.view_as_complex(torch.rand(b, n, 2, generator=g, device="cuda") * 2 - 1)
    y = ops.c2c(x, sign, scale=1.0)
    z = ops.c2c(x, sign, scale=0.375)
    padded = torch.empty(b, n + 2, dtype=torch.complex64, device="cuda")
    ops.c2c_rows(x, sign, out=padded[:, :n])
    torch.cuda.synchronize()
    pick = sorted({0, 1, b // 2, b - 2, b - 1, *range(3, b, max(1, b // 12))})
    want = oracle.c2c_f64(_rows(x, pick, n), n, sign)
    assert oracle.rel_l2_rows(_rows(y, pick, n), want) <= REL_L2
    assert oracle.rel_l2_rows(_rows(padded[:, :n], pick, n), want) <= REL_L2
    # the scale is one FP32 product in the last store
    assert np.array_equal(_rows(z, list(range(b)), n), _rows(y, list(range(b)), n) * np.float32(0.375))
