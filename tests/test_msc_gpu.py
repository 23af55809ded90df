"""The GPU reading of a .grad as extractmsc reads it (msceer_msc_base: nodes,
base basins, base mountains), bit-exact against the reference's own
Morse-Smale complex class on the lower-star goldens and against the oracle
on GPU-made .grad files of larger seeded volumes."""
import ctypes
import sys

import numpy as np
import pytest

import oracle_lib
from golden import load_msc, msc_case_names
from msceer_amd import hipmem, lstar, msc, native, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("name", msc_case_names())
def test_reference_goldens(ctx, name):
    f, grad, basins, mounts, counts = load_msc(name)
    b, m, c = msc.msc_base(grad, f.shape, ctx=ctx)
    assert (c == counts).all(), (c, counts)
    assert (b == basins).all(), int((b != basins).sum())
    assert (m == mounts).all(), int((m != mounts).sum())


@pytest.mark.parametrize("shape,seed,kind", [((96, 112, 128), 41, "noise"), ((128, 128, 128), 42, "gauss"),
                                             ((7, 300, 33), 43, "noise")])
def test_gpu_grad_against_oracle(ctx, shape, seed, kind):
    f = (synth.smoothed_noise(shape, seed, 2.0) if kind == "noise"
         else synth.gaussian_mixture(shape, seed, 40, 3.0, 10.0, -1.0, 1.0)).astype(np.float32)
    g = lstar.steepest_lstar_grad(f, ctx=ctx).ravel()
    print(f"{shape} {kind}", flush=True)
    sys.stdout.flush()
    b, m, c = msc.msc_base(g, f.shape, ctx=ctx)
    rb, rm, rc = oracle_lib.msc_base(g, f.shape)
    assert (c == rc).all()
    assert (b == rb).all(), int((b != rb).sum())
    assert (m == rm).all(), int((m != rm).sum())


def test_device_pointers_and_one_output(ctx):
    f, grad, basins, mounts, counts = load_msc("noise_48x97x31")
    Z, Y, X = f.shape
    dg = hipmem.DeviceBuffer(grad.size)
    dg.upload(grad)
    dm = hipmem.DeviceBuffer(4 * f.size)
    dm.fill(0x7F)
    hipmem.synchronize()
    native.check(native.lib().msceer_msc_base(ctx.handle, ctypes.c_void_p(dg.addr), X, Y, Z, None,
                                              ctypes.c_void_p(dm.addr), None, native.DEVICE_PTRS), "msceer_msc_base")
    hipmem.synchronize()
    m = dm.download(np.int32, f.size).reshape(f.shape)
    assert (m == mounts).all()


@pytest.mark.parametrize("shape", [(2, 2, 2), (2, 2, 70), (2, 70, 2), (70, 2, 2), (5, 4, 65), (4, 9, 64), (6, 5, 129)])
def test_tile_edges_against_oracle(ctx, shape):
    # paths followed inside 64x4x4 tiles, extents of one hex (coinciding strides) among them
    f = synth.Stream(44).normal(int(np.prod(shape))).reshape(shape).astype(np.float32)
    g = oracle_lib.steepest_grad(f)
    print(shape, flush=True)
    b, m, c = msc.msc_base(g, shape, ctx=ctx)
    rb, rm, rc = oracle_lib.msc_base(g, shape)
    assert (c == rc).all()
    assert (b == rb).all(), int((b != rb).sum())
    assert (m == rm).all(), int((m != rm).sum())


def test_thin_volume_of_more_tiles_than_a_grid_holds(ctx):
    """2 x 4100 x 65536 vertices: 1025 x 16384 tiles of 256 threads.  Every
    vertex is paired towards lower z, so a column's basin is its lowest vertex,
    the only critical cells there are."""
    X, Y, Z = 2, 4100, 65536
    plane = (2 * X - 1) * (2 * Y - 1)
    dg = hipmem.DeviceBuffer(plane * (2 * Z - 1))
    db = hipmem.DeviceBuffer(4 * X * Y * Z)
    dg.fill(1)  # assigned, paired towards higher x
    db.fill(0x7F)
    hipmem.synchronize()
    layer = np.full((2 * Y - 1, 2 * X - 1), 1, np.uint8)
    for z in range(Z):
        if z < 2:
            layer[::2, ::2] = 1 | (7 if z == 0 else 5) << 2
        dg.upload_at(2 * z * plane, layer)
    counts = (ctypes.c_int64 * 4)()
    print("thin volume: uploaded", flush=True)
    native.check(native.lib().msceer_msc_base(ctx.handle, ctypes.c_void_p(dg.addr), X, Y, Z, ctypes.c_void_p(db.addr),
                                              None, ctypes.cast(counts, ctypes.c_void_p), native.DEVICE_PTRS), "msc")
    assert list(counts) == [X * Y, 0, 0, 0]
    expect = np.tile(np.arange(X * Y, dtype=np.int32), 4096)
    for z in range(0, Z, 4096):
        assert np.array_equal(db.download_at(4 * X * Y * z, np.int32, expect.size), expect), z
