"""Ascending-manifold dimension on bit planes (ldir.hip) at the edges of its
words and tiles: x extents around one and two 64-vertex words, volumes too
narrow in x whose words run along y or z, y and z around the 4-row and 16-row
tiles, two-vertex slabs, long ways through every tile (a
snake), against the oracle's `.grad`; exact.  One volume, all in one batch, and
into a buffer that starts at an odd byte."""
import numpy as np
import pytest

import oracle_lib
from msceer_amd import batch, hipmem, lstar, native, synth

pytestmark = pytest.mark.gpu

# (Z, Y, X)
SHAPES = [(2, 2, 2), (3, 4, 5), (5, 3, 63), (4, 5, 64), (6, 2, 65), (17, 16, 33), (16, 17, 129), (2, 33, 127),
          (65, 18, 3), (3, 130, 17), (33, 34, 31), (128, 2, 2)]


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


def _snake(shape):
    # values rise along a way that runs through every row
    f = np.arange(int(np.prod(shape)), dtype=np.float32).reshape(shape)
    f[:, 1::2] = f[:, 1::2, ::-1]
    f[1::2] = f[1::2, ::-1, ::-1]
    return np.ascontiguousarray(f)


def _field(kind, shape):
    n = int(np.prod(shape))
    if kind == "noise":
        return synth.Stream(31).normal(n).reshape(shape).astype(np.float32)
    if kind == "smooth":
        return synth.smoothed_noise(shape, 32, 2.0)
    if kind == "ties":
        return np.floor(synth.Stream(33).uniform(n) * 3).reshape(shape).astype(np.float32)
    return _snake(shape) if kind == "snake" else -_snake(shape)


KINDS = ["noise", "smooth", "ties", "snake", "down"]


@pytest.mark.parametrize("kind", KINDS)
def test_single_volumes(ctx, kind):
    for shape in SHAPES:
        print("ldir", kind, shape, flush=True)
        f = _field(kind, shape)
        g = lstar.steepest_lstar_grad(f, ctx).ravel()
        assert np.array_equal(g, oracle_lib.steepest_grad(f).ravel()), (kind, shape)


def test_one_batch(ctx):
    print("ldir batch", flush=True)
    fs = [_field(k, s) for s in SHAPES for k in KINDS]
    grads, _, _ = batch.run_batch_grad(fs, ctx=ctx)
    for f, g in zip(fs, grads):
        assert np.array_equal(g.ravel(), oracle_lib.steepest_grad(f).ravel()), f.shape


@pytest.mark.parametrize("shape", [(5, 6, 65), (9, 4, 64), (40, 5, 6)])
def test_output_at_an_odd_byte(ctx, shape):
    print("ldir odd byte", shape, flush=True)
    f = _field("noise", shape)
    ref = oracle_lib.steepest_grad(f).ravel()
    vals, out = hipmem.DeviceBuffer(f.nbytes), hipmem.DeviceBuffer(ref.size + 8)
    vals.upload(f)
    out.fill(0xA5)
    lstar.steepest_lstar_grad_device(ctx, vals.addr, shape[2], shape[1], shape[0], out.addr + 3)
    got = out.download(np.uint8, ref.size + 8)
    assert np.array_equal(got[3:3 + ref.size], ref)
    assert (got[:3] == 0xA5).all() and (got[3 + ref.size:] == 0xA5).all()
