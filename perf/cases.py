"""The calls whose speed counts, as a user's program makes them.

One context is kept for all of them, as a program that works through volumes
keeps one.  Volumes are device tensors unless a case says otherwise: the
fields are those of the package's own workloads (Gaussian mixtures, white
noise smoothed by a Gaussian, both made here on the GPU from the seed), the
parameters those of its benchmark (squared step error 1e-3, gradient 1e-6,
4096 steps).  Outputs are bytes and vertex ids, compared as they are; only
the classifier's probabilities are computed numbers with an exact value.
"""
import ctypes
import math
import os
import random

import numpy as np
import torch

from msceer_amd import batch, learned, lstar, native

ERR, GTHR, ITERS = 1e-3, 1e-6, 4096
DEV = "cuda"
WEIGHTS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "msceer_amd", "weights",
                       "sepnet.npz")

_kept = {}


def _ctx():
    """The context a program keeps across its calls."""
    if "ctx" not in _kept:
        _kept["ctx"] = native.Context(0)
    return _kept["ctx"]


def _net():
    """The trained classifier, loaded once."""
    if "net" not in _kept:
        net = learned.SeparatrixNet(_ctx())
        net.load()
        _kept["net"] = net
    return _kept["net"]


# ---------------------------------------------------------------------------
# cases


def listed():
    return [
        # a small volume alone: launches and waits are most of the call
        {"name": "grad_64", "kind": "grad", "x": 64, "y": 64, "z": 64, "field": "bumps", "sigma": 0.0},
        # an ordinary ragged volume from and to the caller's numpy arrays, as
        # the command-line program and the Python mirror do it
        {"name": "grad_host_131x97x48", "kind": "grad_host", "x": 131, "y": 97, "z": 48, "field": "noise",
         "sigma": 2.0},
        # the large volume of dense critical points
        {"name": "grad_512", "kind": "grad", "x": 512, "y": 512, "z": 512, "field": "noise", "sigma": 2.0},
        # many uneven volumes (sides 32 to 160) resident on the card
        {"name": "batch_grad_96", "kind": "batch_grad", "count": 96, "shapes": 1},
        # accurate labels and .grad of many uneven host volumes
        {"name": "batch_labels_16", "kind": "batch_labels", "count": 16, "shapes": 2},
        # accurate ascending labels and the conforming .grad: small, the
        # benchmark's labelling volume, a large ragged one of noise
        {"name": "labels_64", "kind": "labels", "x": 64, "y": 64, "z": 64, "field": "mixture", "sigma": 0.0,
         "presimp": 0.0, "need": native.NEED_ASC2},
        {"name": "labels_256", "kind": "labels", "x": 256, "y": 256, "z": 256, "field": "mixture", "sigma": 0.0,
         "presimp": 0.0, "need": native.NEED_ASC2},
        {"name": "labels_500x380x260", "kind": "labels", "x": 500, "y": 380, "z": 260, "field": "noise",
         "sigma": 2.5, "presimp": 0.0, "need": native.NEED_ASC2},
        # the accurate 1-manifolds of both families on the labelling volume
        {"name": "lines_256", "kind": "labels", "x": 256, "y": 256, "z": 256, "field": "mixture", "sigma": 0.0,
         "presimp": 0.0, "need": native.NEED_ASC1 | native.NEED_DSC1},
        # every accuracy branch at once, with a persistence threshold
        {"name": "all_branches_160x144x131", "kind": "labels", "x": 160, "y": 144, "z": 131, "field": "noise",
         "sigma": 2.5, "presimp": 0.05,
         "need": native.NEED_ASC1 | native.NEED_DSC1 | native.NEED_ASC2 | native.NEED_DSC2},
        # the reading of a .grad as a Morse-Smale complex base
        {"name": "msc_base_256", "kind": "msc", "x": 256, "y": 256, "z": 256, "field": "noise", "sigma": 2.0},
        # the near-separatrix classifier on the volume size of its evaluation
        {"name": "predict_256x192x128", "kind": "predict", "x": 256, "y": 192, "z": 128, "field": "noise",
         "sigma": 2.5},
    ]


def _side(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _sides(rng, lo, hi, most):
    """Three sides in [lo, hi], spread over their logarithm, with at most `most` vertices."""
    while True:
        s = [_side(rng, lo, hi) for _ in range(3)]
        if s[0] * s[1] * s[2] <= most:
            return {"x": s[0], "y": s[1], "z": s[2]}


def _field(rng):
    if rng.random() < 0.5:
        return {"field": "mixture", "sigma": 0.0}
    return {"field": "noise", "sigma": round(rng.uniform(1.5, 3.0), 2)}


def draw(rng: random.Random):
    kind = rng.choice(["grad", "grad", "grad_host", "batch_grad", "batch_labels", "labels", "labels", "lines",
                       "branches", "msc", "predict"])
    if kind == "grad":
        return {"kind": kind, **_sides(rng, 24, 512, 400 ** 3), **_field(rng)}
    if kind == "grad_host":
        return {"kind": kind, **_sides(rng, 24, 192, 128 ** 3), **_field(rng)}
    if kind == "batch_grad":
        return {"kind": kind, "count": rng.randint(8, 96), "shapes": rng.randint(10, 1 << 20)}
    if kind == "batch_labels":
        return {"kind": kind, "count": rng.randint(4, 16), "shapes": rng.randint(10, 1 << 20)}
    if kind == "labels":
        return {"kind": "labels", **_sides(rng, 32, 400, 256 ** 3), **_field(rng), "presimp": rng.choice([0.0, 0.0, 0.05]),
                "need": native.NEED_ASC2}
    if kind == "lines":
        return {"kind": "labels", **_sides(rng, 48, 256, 160 ** 3), "field": "mixture", "sigma": 0.0, "presimp": 0.0,
                "need": rng.choice([native.NEED_ASC1, native.NEED_DSC1, native.NEED_ASC1 | native.NEED_DSC1])}
    if kind == "branches":
        return {"kind": "labels", **_sides(rng, 48, 192, 128 ** 3), **_field(rng), "presimp": rng.choice([0.0, 0.05]),
                "need": rng.choice([native.NEED_DSC2, native.NEED_ASC2 | native.NEED_DSC2,
                                    native.NEED_ASC1 | native.NEED_ASC2,
                                    native.NEED_ASC1 | native.NEED_DSC1 | native.NEED_ASC2 | native.NEED_DSC2])}
    return {"kind": kind, **_sides(rng, 32, 320, 200 ** 3), **_field(rng)}


# ---------------------------------------------------------------------------
# fields


def _smooth(f, sigma, dim):
    """Gaussian filter along one axis (truncated at 4 sigma, mirrored edges)."""
    r = int(4.0 * sigma + 0.5)
    n = f.shape[dim]
    w = [math.exp(-0.5 * (k / sigma) ** 2) for k in range(r + 1)]
    total = w[0] + 2.0 * sum(w[1:])
    at = torch.arange(-r, n + r, device=f.device)
    period = max(1, 2 * (n - 1))
    at = at.remainder(period)
    at = torch.where(at >= n, period - at, at)
    g = f.index_select(dim, at)
    out = g.narrow(dim, r, n) * (w[0] / total)
    for k in range(1, r + 1):
        out.add_(g.narrow(dim, r - k, n), alpha=w[k] / total).add_(g.narrow(dim, r + k, n), alpha=w[k] / total)
    return out


def _noise(shape, sigma, gen):
    f = torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32)
    for dim in range(3):
        f = _smooth(f, sigma, dim)
    return f


def _mixture(shape, gen, count, lo, hi, sine=0.0, noise=0.0):
    Z, Y, X = shape
    p = torch.rand((5, count), generator=gen, device="cpu", dtype=torch.float64)
    k = 0.05 + 0.15 * torch.rand(3, generator=gen, device="cpu", dtype=torch.float64)
    cx, cy, cz = p[0] * (X - 1), p[1] * (Y - 1), p[2] * (Z - 1)
    sig, amp = lo + (hi - lo) * p[3], 2.0 * p[4] - 1.0
    axis = [torch.arange(n, dtype=torch.float64) for n in (X, Y, Z)]
    inv = (-0.5 / (sig * sig))[:, None]
    ex = torch.exp(inv * (axis[0][None] - cx[:, None]) ** 2).to(DEV)
    ey = torch.exp(inv * (axis[1][None] - cy[:, None]) ** 2).to(DEV)
    ez = (amp[:, None] * torch.exp(inv * (axis[2][None] - cz[:, None]) ** 2)).to(DEV)
    f = torch.zeros(shape, device=DEV, dtype=torch.float64)
    for g in range(count):
        f.addcmul_(ez[g][:, None, None] * ey[g][None, :, None], ex[g][None, None, :])
    if sine:
        sx, sy, sz = (torch.sin(k[i] * axis[i]).to(DEV) for i in range(3))
        f.addcmul_(sz[:, None, None] * sy[None, :, None], sx[None, None, :], value=sine)
    if noise:
        f += noise * (2.0 * torch.rand((Z, Y, X), generator=torch.Generator(DEV).manual_seed(gen.initial_seed()),
                                       device=DEV, dtype=torch.float64) - 1.0)
    return f.float()


def _volume(shape, field, sigma, seed):
    """A (Z, Y, X) float32 device tensor."""
    if field == "noise":
        return _noise(shape, sigma, torch.Generator(DEV).manual_seed(seed))
    gen = torch.Generator("cpu").manual_seed(seed)
    if field == "bumps":
        return _mixture(shape, gen, 32, 3.0, 10.0, noise=1e-3)
    n = max(4, round(200 * shape[0] * shape[1] * shape[2] / 256 ** 3))
    return _mixture(shape, gen, n, 4.0, 16.0, sine=0.05)


def _shape(case):
    return case["z"], case["y"], case["x"]


def _cells(shape):
    return (2 * shape[0] - 1) * (2 * shape[1] - 1) * (2 * shape[2] - 1)


def _shapes(case):
    """The shapes and fields of a batch: sides 32 to 160, noise and mixtures by turns."""
    r = random.Random(case["shapes"])
    return [(tuple(r.randint(32, 160) for _ in range(3)), "noise" if i % 2 else "mixture",
             round(r.uniform(1.5, 3.0), 2)) for i in range(case["count"])]


# ---------------------------------------------------------------------------
# one call


def prepare(case, seed):
    kind = case["kind"]
    ctx = _ctx()
    state = {"kind": kind, "ctx": ctx}
    if kind in ("batch_grad", "batch_labels"):
        todo = _shapes(case)
        vols = [_volume(s, f, sg, seed * 4096 + i) for i, (s, f, sg) in enumerate(todo)]
        if kind == "batch_labels":
            state["volumes"] = [v.cpu().numpy() for v in vols]
            return state
        # the .grads in one allocation, each from a 256-byte boundary on
        at, total = [], 0
        for s, _, _ in todo:
            at.append(total)
            total += (_cells(s) + 255) // 256 * 256
        state["volumes"] = vols
        state["grad"] = torch.zeros(total, dtype=torch.uint8, device=DEV)
        state["table"] = batch.volume_table([s for s, _, _ in todo], [v.data_ptr() for v in vols],
                                            [state["grad"].data_ptr() + o for o in at])
        return state
    shape = _shape(case)
    V, C = shape[0] * shape[1] * shape[2], _cells(shape)
    f = _volume(shape, case["field"], case["sigma"], seed)
    state["shape"] = shape
    if kind == "grad_host":
        state["values"] = f.cpu().numpy()
        return state
    state["values"] = f
    if kind == "grad":
        state["grad"] = torch.empty(C, dtype=torch.uint8, device=DEV)
    elif kind == "labels":
        need = case["need"]
        state["need"], state["presimp"] = need, case["presimp"]
        state["stats"] = native.LabelStats()
        state["grad"] = torch.empty(C, dtype=torch.uint8, device=DEV)
        state["restriction"] = torch.empty(C, dtype=torch.int8, device=DEV) if need != native.NEED_ASC2 else None
        state["labels"] = torch.empty(V, dtype=torch.int32, device=DEV) if need & native.NEED_ASC2 else None
        state["labels_dsc"] = torch.empty(V, dtype=torch.int32, device=DEV) if need & native.NEED_DSC2 else None
    elif kind == "msc":
        state["grad"] = torch.empty(C, dtype=torch.uint8, device=DEV)
        torch.cuda.synchronize()
        lstar.steepest_lstar_grad_device(ctx, f.data_ptr(), shape[2], shape[1], shape[0], state["grad"].data_ptr())
        state["basins"] = torch.empty(V, dtype=torch.int32, device=DEV)
        state["mounts"] = torch.empty(V, dtype=torch.int32, device=DEV)
        state["counts"] = np.zeros(4, np.int64)
    else:
        state["net"] = _net()
        state["prob"] = torch.empty(V, dtype=torch.float32, device=DEV)
    return state


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "grad_host":
        return lstar.steepest_lstar_grad(state["values"], ctx)
    if kind == "batch_labels":
        grads, labels, _ = batch.run_batch(state["volumes"], labels=True, ctx=ctx)
        return {"grads": grads, "labels": labels}
    lib = native.lib()
    if kind == "batch_grad":
        native.check(lib.msceer_batch_grad(ctx.handle, state["table"], len(state["table"]), 0, native.DEVICE_PTRS),
                     "msceer_batch_grad")
        return state["grad"]
    Z, Y, X = state["shape"]
    values = state["values"]
    if kind == "grad":
        lstar.steepest_lstar_grad_device(ctx, values.data_ptr(), X, Y, Z, state["grad"].data_ptr())
        return state["grad"]
    if kind == "labels":
        out = {k: state[k] for k in ("grad", "labels", "labels_dsc", "restriction")}
        if state["need"] == native.NEED_ASC2:
            rc = lib.msceer_ondemand_asc(ctx.handle, _ptr(values), X, Y, Z, ERR, GTHR, ITERS, state["presimp"], None,
                                         _ptr(out["grad"]), _ptr(out["labels"]), ctypes.byref(state["stats"]),
                                         native.DEVICE_PTRS)
        else:
            rc = lib.msceer_ondemand2(ctx.handle, _ptr(values), X, Y, Z, ERR, GTHR, ITERS, state["presimp"],
                                      state["need"], None, _ptr(out["grad"]), _ptr(out["labels"]),
                                      _ptr(out["labels_dsc"]), _ptr(out["restriction"]),
                                      ctypes.byref(state["stats"]), native.DEVICE_PTRS)
        native.check(rc, "msceer_ondemand")
        return {k: v for k, v in out.items() if v is not None}
    if kind == "msc":
        native.check(lib.msceer_msc_base(ctx.handle, _ptr(state["grad"]), X, Y, Z, _ptr(state["basins"]),
                                         _ptr(state["mounts"]), state["counts"].ctypes.data_as(ctypes.c_void_p),
                                         native.DEVICE_PTRS), "msceer_msc_base")
        return {"basins": state["basins"], "mounts": state["mounts"], "counts": state["counts"]}
    native.check(lib.msceer_cnn_predict(ctx.handle, state["net"]._h, _ptr(values), X, Y, Z, _ptr(state["prob"]),
                                        native.DEVICE_PTRS), "msceer_cnn_predict")
    return state["prob"]


def work(case):
    """Values read once, outputs written once; the classifier's multiplications."""
    if case["kind"] in ("batch_grad", "batch_labels"):
        per = 4 + (4 if case["kind"] == "batch_labels" else 0)
        return {"bytes": sum(per * s[0] * s[1] * s[2] + _cells(s) for s, _, _ in _shapes(case)), "flops": 0}
    shape = _shape(case)
    V, C = shape[0] * shape[1] * shape[2], _cells(shape)
    if case["kind"] == "msc":
        return {"bytes": C + 8 * V, "flops": 0}
    if case["kind"] == "predict":
        return {"bytes": 8 * V, "flops": 2 * V * (27 * 16 + 27 * 16 * 32 + 27 * 32 * 16 + 16)}
    nbytes = 4 * V + C
    if case["kind"] == "labels":
        need = case["need"]
        nbytes += 4 * V * (bool(need & native.NEED_ASC2) + bool(need & native.NEED_DSC2))
        nbytes += C if need != native.NEED_ASC2 else 0
    return {"bytes": nbytes, "flops": 0}


# ---------------------------------------------------------------------------
# the classifier in 64 bits


def _window_sum(a, r=4):
    for dim in range(a.dim()):
        n = a.shape[dim]
        s = a.clone()
        for k in range(1, min(r, n - 1) + 1):
            s.narrow(dim, 0, n - k).add_(a.narrow(dim, k, n - k))
            s.narrow(dim, k, n - k).add_(a.narrow(dim, 0, n - k))
        a = s
    return a


def _conv(a, w, bias):
    """a (C, Z, Y, X), w (27, out, in): tap t reads (x + t % 3 - 1, y + t / 3 % 3 - 1, z + t / 9 - 1), zero outside."""
    Z, Y, X = a.shape[1:]
    out = bias[:, None, None, None].expand(-1, Z, Y, X).clone()
    for t in range(27):
        d = (t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1)
        to = [slice(max(0, -k), n - max(0, k)) for k, n in zip(d, (Z, Y, X))]
        of = [slice(max(0, k), n - max(0, -k)) for k, n in zip(d, (Z, Y, X))]
        src = a[(slice(None), *of)]
        out[(slice(None), *to)] += (w[t] @ src.reshape(a.shape[0], -1)).reshape(w.shape[1], *src.shape[1:])
    return out.clamp_(min=0.0)


def exact(case, seed):
    if case["kind"] != "predict":
        return None  # bytes and vertex ids
    shape = _shape(case)
    f = _volume(shape, case["field"], case["sigma"], seed).double()
    c = _window_sum(torch.ones_like(f))
    mean = _window_sum(f) / c
    var = (_window_sum(f * f) / c - mean * mean).clamp_(min=0.0)
    a = ((f - mean) / (var.sqrt() + 1e-6))[None]
    with np.load(WEIGHTS) as d:
        p = torch.from_numpy(d["params"].astype(np.float64)).to(DEV)
    at = 0
    for cin, cout in ((1, 16), (16, 32), (32, 16)):
        w = p[at:at + 27 * cout * cin].reshape(27, cout, cin)
        at += w.numel()
        a = _conv(a, w, p[at:at + cout])
        at += cout
    z = (p[at:at + 16] @ a.reshape(16, -1)) + p[at + 16]
    return torch.sigmoid(z)
