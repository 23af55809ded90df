"""Certain regions of the labelling (chains and flood, certain.hip) at the
edges of their tiles: x extents around one and two 64-vertex words, y and z
around the 4-row chain tiles and the 16-row flood tiles, two-vertex slabs, long
monotone ways (a snake through every tile), ties and signed zeros, in both
orders, against the defining rule taken vertex by vertex; exact."""
import ctypes
import sys

import numpy as np
import pytest

import oracle_lib
from msceer_amd import hipmem, labels, native, synth

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 5, 63), (4, 4, 64), (5, 3, 65), (16, 17, 33), (17, 16, 64), (33, 15, 129), (2, 40, 191)]


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def _noise(shape, seed):
    return synth.Stream(seed).normal(int(np.prod(shape))).reshape(shape).astype(np.float32)


def _snake(shape):
    # values rise along a way that runs through every row: one long chain
    Z, Y, X = shape
    f = np.arange(Z * Y * X, dtype=np.float32).reshape(shape)
    f[:, 1::2] = f[:, 1::2, ::-1]
    f[1::2] = f[1::2, ::-1, ::-1]
    return np.ascontiguousarray(f)


def _ties(shape, seed):
    u = synth.Stream(seed).uniform(int(np.prod(shape))).reshape(shape)
    f = np.floor(u * 4).astype(np.float32) - 1.0
    f[u < 0.1] = -0.0
    return f


FIELDS = {"noise": lambda s: _noise(s, 71), "smooth": lambda s: synth.smoothed_noise(s, 72, 2.0),
          "snake": _snake, "ties": lambda s: _ties(s, 73)}


def _rule(f, seed, lab, desc):
    """The defining rule, vertex by vertex: the label all earlier neighbours share."""
    Z, Y, X = f.shape
    V = f.size
    order = np.lexsort((np.arange(V), f.ravel()))
    rank = np.empty(V, np.int64)
    rank[order] = np.arange(V)
    if desc:
        order, rank = order[::-1], V - 1 - rank
    lab = np.where(seed, lab, -1)
    for v in order:
        if seed[v]:
            continue
        x, y, z = v % X, (v // X) % Y, v // (X * Y)
        ls = [lab[v + d] for d, ok in ((1, x < X - 1), (-1, x > 0), (X, y < Y - 1), (-X, y > 0),
                                       (X * Y, z < Z - 1), (-X * Y, z > 0)) if ok and rank[v + d] < rank[v]]
        if ls and ls[0] != -1 and all(q == ls[0] for q in ls):
            lab[v] = ls[0]
    return lab


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", sorted(FIELDS))
def test_ascending_regions_follow_the_rule(ctx, shape, kind):
    print(f"certain asc {kind} {shape}", flush=True)
    f = FIELDS[kind](shape)
    _, lab, _ = labels.ondemand_asc(f, ctx=ctx, stop="regions")
    lab = lab.ravel()
    Z, Y, X = shape
    seed = (((oracle_lib.lstar_pairs(f).reshape(2 * Z - 1, 2 * Y - 1, 2 * X - 1)[::2, ::2, ::2] >> 2) & 7) == 7).ravel()
    # (the seeds' names come out of the simplification, which is not tested here)
    assert (lab[seed] >= 0).all()
    assert (lab == _rule(f, seed, lab, False)).all()


def _maxima(f):
    """The highest vertices of the critical hexes."""
    Z, Y, X = f.shape
    base = oracle_lib.lstar_pairs(f).reshape(2 * Z - 1, 2 * Y - 1, 2 * X - 1)
    order = np.lexsort((np.arange(f.size), f.ravel()))
    rank = np.empty(f.size, np.int64)
    rank[order] = np.arange(f.size)
    seed = np.zeros(f.size, bool)
    r3 = rank.reshape(Z, Y, X)
    for z, y, x in np.argwhere(((base[1::2, 1::2, 1::2] >> 2) & 7) == 7):
        seed[order[r3[z:z + 2, y:y + 2, x:x + 2].max()]] = True
    return seed


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["noise", "smooth", "snake"])
def test_descending_regions_follow_the_rule(ctx, shape, kind):
    print(f"certain desc {kind} {shape}", flush=True)
    sys.stdout.flush()
    f = FIELDS[kind](shape)
    Z, Y, X = f.shape
    dv = hipmem.DeviceBuffer(f.nbytes)
    dv.upload(f)
    dl = hipmem.DeviceBuffer(4 * f.size)
    st = native.LabelStats()
    native.check(native.lib().msceer_ondemand2(ctx.handle, ctypes.c_void_p(dv.addr), X, Y, Z, 1e-3, 1e-6, 64, 0.0,
                                               native.NEED_DSC2, None, None, None, ctypes.c_void_p(dl.addr), None,
                                               ctypes.byref(st), native.DEVICE_PTRS | native.STOP_REGIONS),
                 "msceer_ondemand2")
    hipmem.synchronize()
    assert (dl.download(np.int32, f.size) == _rule(f, _maxima(f), np.arange(f.size), True)).all()


def test_more_tiles_than_one_launch_takes(ctx):
    """2 x 2100 x 8320 vertices, 525 x 2080 tiles in two launches: noise that
    repeats every 16 layers, so its regions repeat too, but for the first and
    the last layers.  Four repeats follow the rule, and all of them are alike."""
    X, Y, P, n = 2, 2100, 16, 520
    one = _noise((P, Y, X), 74)
    print("certain, two launches", flush=True)

    def regions(k):
        f = np.tile(one, (k, 1, 1))
        _, lab, _ = labels.ondemand_asc(f, ctx=ctx, stop="regions")
        return f, lab

    f, few = regions(4)
    Z = 4 * P
    seed = (((oracle_lib.lstar_pairs(f).reshape(2 * Z - 1, 2 * Y - 1, 2 * X - 1)[::2, ::2, ::2] >> 2) & 7) == 7).ravel()
    assert (few.ravel() == _rule(f, seed, few.ravel(), False)).all()
    _, lab = regions(n)
    step = P * X * Y  # ids of one repeat
    lab = lab.reshape(n, P, Y, X)
    for k in range(n):
        at = min(k, 1) if k < n - 1 else 3  # the first, an inner one, the last
        assert ((lab[k] == -1) == (few.reshape(4, P, Y, X)[at] == -1)).all(), k
        known = lab[k] >= 0
        assert (lab[k][known] - k * step == few.reshape(4, P, Y, X)[at][known] - at * step).all(), k
