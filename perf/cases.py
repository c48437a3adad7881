"""Workloads of the library's public Python entry points, with their sizes, inputs and 64-bit results.

listed() are the fixed ones; draw() gives more of the same kinds:

  c2c       complex transform along the last axis (ops.c2c): both directions, every norm, both layouts
  rfft      real to half spectrum (ops.rfft)
  irfft     half spectrum to real (ops.irfft)
  fft2      2-D complex transform (ops.fft2)
  columns   complex transform along the axis before the last (ops.fft_columns)
  group     many uneven requests in one launch (group.Group)
  spectral  spectral convolution layer, forward and backward (spectral.spectral_conv1d)
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "ascend-fft_amd"))

from bfly import KIND_C2C, group, ops, spectral  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # one small request of a serving loop: a launch and its latency
        {"name": "c2c_1024x64", "kind": "c2c", "n": 1024, "batch": 64, "sign": -1, "norm": "", "layout": "complex"},
        # a spectrum taken back to the time domain with numpy's 1/n: a mid-size, ragged batch
        {"name": "ifft_512x1500", "kind": "c2c", "n": 512, "batch": 1500, "sign": 1, "norm": "backward",
         "layout": "complex"},
        # the library's headline workload: a full batch of interleaved rows
        {"name": "c2c_4096x4096", "kind": "c2c", "n": 4096, "batch": 4096, "sign": -1, "norm": "",
         "layout": "interleaved"},
        # long transforms: pulse compression and spectrum analysis lengths, whole and ragged batches
        {"name": "c2c_16384x1000", "kind": "c2c", "n": 16384, "batch": 1000, "sign": -1, "norm": "",
         "layout": "interleaved"},
        {"name": "c2c_32768x256", "kind": "c2c", "n": 32768, "batch": 256, "sign": -1, "norm": "",
         "layout": "interleaved"},
        {"name": "c2c_65536x64", "kind": "c2c", "n": 65536, "batch": 64, "sign": -1, "norm": "",
         "layout": "interleaved"},
        # real signals to half spectra, a full batch, and back from a mid-size ragged one
        {"name": "rfft_4096x4096", "kind": "rfft", "n": 4096, "batch": 4096},
        {"name": "irfft_2048x999", "kind": "irfft", "n": 2048, "batch": 999},
        # images / range-Doppler maps
        {"name": "fft2_1024x1024x16", "kind": "fft2", "n1": 1024, "n2": 1024, "batch": 16, "sign": -1},
        # Doppler transform along the pulses of a data cube whose range gates are no power of two
        {"name": "columns_512x1001x24", "kind": "columns", "n": 512, "ncols": 1001, "batch": 24, "sign": -1},
        # a serving step: 512 requests of all lengths, complex and real, in one launch
        {"name": "group_512req", "kind": "group", "count": 512, "spec_seed": 3, "n_min": 64, "n_max": 8192,
         "batch_max": 256, "dynamic": 1},
        # a training step of the spectral layer of a neural operator
        {"name": "spectral_64x128x4096", "kind": "spectral", "B": 64, "c_in": 128, "c_out": 128, "n": 4096,
         "modes": 256},
    ]


def _log_int(rng, lo, hi):
    """An integer of lo..hi, uniform over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _pow2(rng, lo, hi):
    return 1 << rng.randint(lo.bit_length() - 1, hi.bit_length() - 1)


def draw(rng):
    kind = rng.choice(["c2c", "c2c", "c2c", "rfft", "irfft", "fft2", "columns", "group", "spectral"])
    most = 1 << 24  # points of the largest plain transform
    if kind == "c2c":
        n = _pow2(rng, 16, 65536)
        return {"kind": kind, "n": n, "batch": _log_int(rng, 1, most // n), "sign": rng.choice([-1, 1]),
                "norm": rng.choice(["", "", "backward", "ortho", "forward"]),
                "layout": rng.choice(["complex", "interleaved"])}
    if kind in ("rfft", "irfft"):
        n = _pow2(rng, 32, 8192)
        return {"kind": kind, "n": n, "batch": _log_int(rng, 1, most // n)}
    if kind == "fft2":
        n1, n2 = _pow2(rng, 16, 4096), _pow2(rng, 16, 4096)
        return {"kind": kind, "n1": n1, "n2": n2, "batch": _log_int(rng, 1, most // (n1 * n2)),
                "sign": rng.choice([-1, 1])}
    if kind == "columns":
        n = _pow2(rng, 16, 4096)
        ncols = _log_int(rng, 1, 4096)
        return {"kind": kind, "n": n, "ncols": ncols, "batch": _log_int(rng, 1, max(1, most // (n * ncols))),
                "sign": rng.choice([-1, 1])}
    if kind == "group":
        return {"kind": kind, "count": _log_int(rng, 8, 256), "spec_seed": rng.randrange(1 << 20),
                "n_min": _pow2(rng, 32, 256), "n_max": _pow2(rng, 1024, 8192), "batch_max": rng.randint(16, 256),
                "dynamic": rng.randint(0, 1)}
    n = _pow2(rng, 256, 8192)
    rows = (1 << 24) // n  # B times the wider side's channels
    c_in, c_out = _log_int(rng, 4, 128), _log_int(rng, 4, 128)
    return {"kind": "spectral", "B": _log_int(rng, 1, min(64, max(1, rows // max(c_in, c_out)))), "c_in": c_in,
            "c_out": c_out, "n": n, "modes": _log_int(rng, 8, min(256, n // 2))}


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _uniform(shape, g):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float32) * 2 - 1


def _complex(shape, g):
    return torch.view_as_complex(_uniform((*shape, 2), g))


def _specs(case):
    return group.uneven_specs(case["count"], case["spec_seed"], case["n_min"], case["n_max"], case["batch_max"])


def _requests(case, seed):
    """The requests of a group, their inputs and outputs cut from one buffer each (256-byte aligned)."""
    reqs = [group.Request(kind, n, b) for kind, n, b in _specs(case)]

    def cut(sizes):
        at, total = [], 0
        for s in sizes:
            at.append(total)
            total += -(-s // 64) * 64
        return at, total

    xs, nx = cut([r.in_floats() for r in reqs])
    ys, ny = cut([r.out_floats() for r in reqs])
    x = _uniform((nx,), _generator(seed))
    y = torch.zeros(ny, device=DEV, dtype=torch.float32)
    for r, i, o in zip(reqs, xs, ys):
        r.x, r.y = x[i:i + r.in_floats()], y[o:o + r.out_floats()]
    return reqs, x, y


def _inputs(case, seed):
    """The input tensors of a case (all kinds but group)."""
    g, kind = _generator(seed), case["kind"]
    if kind == "c2c":
        n, b = case["n"], case["batch"]
        return (_complex((b, n), g) if case["layout"] == "complex" else _uniform((b, 2 * n), g),)
    if kind == "rfft":
        return (_uniform((case["batch"], case["n"]), g),)
    if kind == "irfft":
        return (_uniform((case["batch"], case["n"] + 2), g),)
    if kind == "fft2":
        return (_complex((case["batch"], case["n1"], case["n2"]), g),)
    if kind == "columns":
        return (_complex((case["batch"], case["n"], case["ncols"]), g),)
    B, ci, co, n, k = (case[f] for f in ("B", "c_in", "c_out", "n", "modes"))
    x = torch.randn((B, ci, n), generator=g, device=DEV)
    w = torch.randn((ci, co, k, 2), generator=g, device=DEV) * (1 / (2 * ci)) ** 0.5
    up = torch.randn((B, co, n), generator=g, device=DEV)
    return x, torch.view_as_complex(w), up


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "group":
        reqs, _, y = _requests(case, seed)
        # what the tuner picks for the serving workload: 512 threads, short requests first, LDS twiddles
        cfg = group.Config(workgroup=512, order=3, dynamic=case["dynamic"], twiddles=1)
        state |= {"group": group.Group(reqs, cfg), "y": y}
    else:
        state["in"] = _inputs(case, seed)
        if case["kind"] == "spectral":
            for t in state["in"][:2]:
                t.requires_grad_(True)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "group":
        state["group"].launch()
        return state["y"]
    if kind == "spectral":
        x, w, up = state["in"]
        y = spectral.spectral_conv1d(x, w)
        gx, gw = torch.autograd.grad(y, (x, w), up)
        return {"y": y.detach(), "gx": gx, "gw": gw}
    (x,) = state["in"]
    if kind == "c2c":
        if case["norm"]:
            return ops.c2c(x, case["sign"], norm=case["norm"])
        return ops.c2c(x, case["sign"], scale=1.0)
    if kind == "rfft":
        return ops.rfft(x)
    if kind == "irfft":
        return ops.irfft(x, case["n"])
    if kind == "fft2":
        return ops.fft2(x, case["sign"])
    return ops.fft_columns(x, case["sign"])


def _c2c_work(points, n):
    return {"bytes": 16 * points, "flops": 5 * points * math.log2(n)}


def _real_work(rows, n):
    return {"bytes": rows * (4 * n + 4 * (n + 2)), "flops": 2.5 * rows * n * math.log2(n)}


def work(case):
    kind = case["kind"]
    if kind == "c2c":
        return _c2c_work(case["n"] * case["batch"], case["n"])
    if kind in ("rfft", "irfft"):
        return _real_work(case["batch"], case["n"])
    if kind == "fft2":
        return _c2c_work(case["n1"] * case["n2"] * case["batch"], case["n1"] * case["n2"])
    if kind == "columns":
        return _c2c_work(case["n"] * case["ncols"] * case["batch"], case["n"])
    if kind == "group":
        parts = [_c2c_work(n * b, n) if k == KIND_C2C else _real_work(b, n) for k, n, b in _specs(case)]
        return {f: sum(p[f] for p in parts) for f in ("bytes", "flops")}
    B, ci, co, n, k = (case[f] for f in ("B", "c_in", "c_out", "n", "modes"))
    # x, w and the output's gradient in; the output and the two gradients out
    return {"bytes": 4 * B * n * (2 * ci + 2 * co) + 2 * 8 * ci * co * k,
            "flops": 3 * 8 * B * ci * co * k + 2 * 2.5 * B * (ci + co) * n * math.log2(n)}


def _exact_c2c(z, sign, norm):
    """numpy's `norm`; "" is the unscaled transform in both directions."""
    if sign < 0:
        return torch.fft.fft(z, norm=norm or "backward")
    return torch.fft.ifft(z, norm=norm or "forward")


def _exact_half(h, n):
    """C2R of interleaved half spectra [..., n+2]: the edge bins' imaginary parts are not read."""
    z = torch.view_as_complex(h.reshape(*h.shape[:-1], n // 2 + 1, 2)).clone()
    z[..., 0].imag.zero_()
    z[..., -1].imag.zero_()
    return torch.fft.irfft(z, n)


def _flat(z):
    return torch.view_as_real(z).reshape(*z.shape[:-1], -1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "group":
        reqs, x, y = _requests(case, seed)
        out = torch.zeros(y.numel(), dtype=torch.float64)
        for r in reqs:
            o, m = r.y.storage_offset(), r.out_floats()
            xi = r.x.cpu().double().reshape(r.batch, -1)
            if r.kind == KIND_C2C:
                z = torch.fft.fft(torch.view_as_complex(xi.reshape(r.batch, r.n, 2)))
            else:
                z = torch.fft.rfft(xi)
            out[o:o + m] = _flat(z).reshape(-1)
        return out
    ins = [t.cpu() for t in _inputs(case, seed)]
    ins = [t.to(torch.complex128 if t.is_complex() else torch.float64) for t in ins]
    if kind == "spectral":
        x, w, up = ins
        n, k = case["n"], case["modes"]
        xm = torch.fft.rfft(x)[..., :k].permute(2, 0, 1).contiguous()   # [K, B, Cin]
        wm = w.permute(2, 0, 1).contiguous()                            # [K, Cin, Cout]
        ym = torch.bmm(xm, wm).permute(1, 2, 0)

        def back(m):  # C2R of the first k bins
            h = torch.zeros(*m.shape[:-1], n // 2 + 1, dtype=torch.complex128)
            h[..., :k] = m
            return torch.fft.irfft(h, n)

        # adjoints: of the C2R, bin j times v_j / n (v = 1 at the edge bins, whose imaginary part is
        # dropped, 2 elsewhere); of the R2C, n times the C2R with weight 1 at the edge bins and 1/2 elsewhere
        v = torch.full((n // 2 + 1,), 2.0, dtype=torch.float64)
        v[0] = v[-1] = 1.0
        gm = torch.fft.rfft(up)[..., :k] * (v[:k] / n)
        gm[..., 0].imag.zero_()
        if k == n // 2 + 1:
            gm[..., -1].imag.zero_()
        gm = gm.permute(2, 0, 1).contiguous()                           # [K, B, Cout]
        gx = torch.bmm(gm, wm.conj().transpose(1, 2).contiguous()).permute(1, 2, 0)
        gw = torch.bmm(xm.conj().transpose(1, 2).contiguous(), gm).permute(1, 2, 0).contiguous()
        return {"y": back(ym), "gx": back(gx / v[:k]) * n, "gw": gw}
    (x,) = ins
    if kind == "c2c":
        if case["layout"] == "complex":
            return _exact_c2c(x, case["sign"], case["norm"])
        z = torch.view_as_complex(x.reshape(case["batch"], case["n"], 2))
        return _flat(_exact_c2c(z, case["sign"], case["norm"]))
    if kind == "rfft":
        return _flat(torch.fft.rfft(x))
    if kind == "irfft":
        return _exact_half(x, case["n"])
    if kind == "fft2":
        return torch.fft.fft2(x) if case["sign"] < 0 else torch.fft.ifft2(x, norm="forward")
    if case["sign"] < 0:
        return torch.fft.fft(x, dim=-2)
    return torch.fft.ifft(x, dim=-2, norm="forward")
