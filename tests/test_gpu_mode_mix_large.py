"""GPU: bfly_mode_mix with more workgroups than one grid dimension holds (2^32
threads): 2^26 modes and a ragged few of one channel and one batch item, where
the product is one complex multiplication per mode."""
import pytest

pytestmark = pytest.mark.gpu


def test_modes_beyond_one_grid_dimension():
    import torch
    from bfly import _lib, ops
    K = (1 << 26) + 5
    print(f"mode_mix K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(11)
    x, w = (torch.view_as_complex(torch.randn(K, 2, generator=g, device="cuda")) for _ in range(2))
    y = ops.mode_mix(_lib.MIX_FORWARD, x.view(1, 1, K), w.view(1, 1, K), 1, 1, 1, K).view(K)
    want = x * w
    # two products and a sum in FP32 each way, values up to about 6^2: 4 roundings of 6e-8
    assert ((y - want).abs() <= 3e-7 * (x.abs() * w.abs())).all()
