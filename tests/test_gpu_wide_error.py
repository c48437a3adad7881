"""GPU: the 32-points-per-thread kernels are no less accurate than the kernels
they run in place of, on the same inputs, against the FP64 oracle: long rows
under AUTO against the one-workgroup and four-step variants, 4096-point
columns in one pass against the two-pass split (which fewer columns run).

The relative L2 error of 2^18 and more independent values scatters by about
1/sqrt(2^19) = 0.14 %; the two errors may differ by three times that."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SCATTER = 1.0042


def _rel(got, want):
    return np.linalg.norm(got - want) / np.linalg.norm(want)


def _host(t, n):
    import torch
    return torch.view_as_real(t).cpu().numpy().reshape(-1, 2 * n)


@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("n,batch,variant", [(8192, 128, "STREAM_LT"), (16384, 160, "FOUR_STEP"),
                                             (16384, 256, "STREAM_LT"), (32768, 129, "FOUR_STEP")])
def test_auto_rows(n, batch, variant, sign):
    import torch
    from bfly import _lib, ops
    lib, s = _lib.hip(), torch.cuda.current_stream().cuda_stream
    print(f"rows n={n} batch={batch} sign={sign}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + batch)
    x = torch.view_as_complex(torch.rand(batch, n, 2, generator=g, device="cuda") * 2 - 1)
    tab, work = ops.table(_lib.KIND_C2C, n, x.device), torch.empty_like(x)
    pick = list(range(0, batch, max(1, batch * n >> 19)))
    want = oracle.c2c_f64(_host(x[pick], n), n, sign)

    def error(v):
        y = torch.empty_like(x)
        assert lib.bfly_c2c_ex(x.data_ptr(), y.data_ptr(), n, batch, sign, v, tab.data_ptr(), work.data_ptr(), s) == 0
        return _rel(_host(y[pick], n), want)

    assert error(_lib.VARIANT_AUTO) <= SCATTER * error(getattr(_lib, f"VARIANT_{variant}"))


@pytest.mark.parametrize("ncols", [128, 125])
def test_one_pass_columns(ncols):
    import torch
    from bfly import ops
    n, batch = 4096, 9  # 1024 columns and more in one call, one matrix at a time in two passes
    print(f"columns n={n} ncols={ncols} batch={batch}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(ncols)
    x = torch.view_as_complex(torch.rand(batch, n, ncols, 2, generator=g, device="cuda") * 2 - 1)
    y, z = ops.fft_columns(x), torch.cat([ops.fft_columns(x[b:b + 1]) for b in range(batch)])
    assert not torch.equal(y, z)  # the two paths
    rows = lambda t: _host(t[::4].transpose(1, 2).contiguous(), n)  # noqa: E731
    want = oracle.c2c_f64(rows(x), n, -1)
    assert _rel(rows(y), want) <= SCATTER * _rel(rows(z), want)
