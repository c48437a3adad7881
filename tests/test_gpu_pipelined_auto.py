"""GPU: bfly_host_pipelined under AUTO runs, on every chunk, what bfly_c2c
runs for a chunk's batch: the results are equal bit for bit, at chunk sizes
where AUTO has a kernel of its own and just below."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pinned", [True, False], ids=["pinned", "pageable"])
@pytest.mark.parametrize("n,chunk,batch", [(8192, 128, 300), (8192, 127, 200), (8192, 0, 300), (16384, 160, 200),
                                           (16384, 256, 300), (32768, 129, 150), (32768, 128, 140)])
def test_auto_equals_bfly_c2c_of_a_chunk(n, chunk, batch, pinned):
    import torch
    from bfly import _lib, ops
    lib, s = _lib.hip(), torch.cuda.current_stream().cuda_stream
    rows = chunk or (8 << 20) // (8 * n)
    print(f"pipelined auto n={n} chunk={rows} batch={batch} pinned={pinned}", flush=True)
    rng = np.random.default_rng(n + chunk)
    x = torch.from_numpy(rng.uniform(-1, 1, (batch, 2 * n)).astype(np.float32))
    hin, hout = (torch.empty(batch, 2 * n, pin_memory=pinned) for _ in range(2))
    hin.copy_(x)
    hout.fill_(float("nan"))
    din, dout = (torch.empty(batch, 2 * n, device="cuda") for _ in range(2))
    work = torch.empty(rows, 2 * n, device="cuda")
    tab = ops.table(_lib.KIND_C2C, n, din.device)
    torch.cuda.synchronize()
    assert lib.bfly_host_pipelined(_lib.KIND_C2C, -1, _lib.VARIANT_AUTO, hin.data_ptr(), hout.data_ptr(), n, batch,
                                   tab.data_ptr(), din.data_ptr(), dout.data_ptr(), work.data_ptr(), chunk, s) == 0
    part, want = x[:rows].cuda(), torch.empty(rows, 2 * n, device="cuda")
    assert lib.bfly_c2c(part.data_ptr(), want.data_ptr(), n, rows, -1, tab.data_ptr(), work.data_ptr(), s) == 0
    torch.cuda.synchronize()
    assert torch.equal(hout[:rows], want.cpu())
    # the last, shorter chunk: the same kernel
    rest = batch - rows
    last = torch.empty(rows, 2 * n, device="cuda")
    part = x[batch - rows:].contiguous().cuda()
    assert lib.bfly_c2c(part.data_ptr(), last.data_ptr(), n, rows, -1, tab.data_ptr(), work.data_ptr(), s) == 0
    torch.cuda.synchronize()
    assert torch.equal(hout[-min(rest, rows):], last.cpu()[-min(rest, rows):])
