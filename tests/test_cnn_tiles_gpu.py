"""The classifier's kernels at the edges of their tiles (32x16 vertices and up
to 8 layers for the convolutions, 64x4 rows for the first, 64x16 and 8 layers
for the normalisation), single vertices along each axis, and in place, against
the CPU oracle (FP64 with BF16 rounding where the kernels store BF16).

Tolerances: probabilities 3e-3 absolute (FP32 accumulation order over 432 to
864 products per output, the odd BF16 rounding flip); the gradient as a whole:
relative L2 error below 3e-2 (two more BF16 roundings)."""
import ctypes

import numpy as np
import pytest

import oracle_lib
from msceer_amd import hipmem, learned, native, synth
from test_oracle_cnn import _params

pytestmark = pytest.mark.gpu

# (Z, Y, X); the last has enough tiles for several layers to a work-group
SHAPES = [(1, 1, 1), (1, 1, 33), (2, 15, 31), (7, 16, 32), (8, 17, 33), (9, 4, 64), (3, 33, 65), (33, 5, 3),
          (17, 130, 1), (19, 260, 257)]


@pytest.fixture(scope="module")
def net():
    c = native.Context(0)
    n = learned.SeparatrixNet(c, seed=3)
    yield n
    n.close()
    c.close()


def _values(shape):
    return synth.Stream(41).normal(int(np.prod(shape))).reshape(shape).astype(np.float32)


@pytest.mark.parametrize("shape", SHAPES)
def test_predict(net, shape):
    print("cnn tiles", shape, flush=True)
    f, p = _values(shape), _params(34)
    net.set_params(p)
    got = net.predict(f)
    err = float(np.abs(got - oracle_lib.cnn_predict(p, f, quant=1)).max())
    print(f"  max error {err:.2e}", flush=True)
    assert err < 3e-3
    # device memory, the probabilities over the values: the same bits
    d = hipmem.DeviceBuffer(f.nbytes)
    d.upload(f)
    native.check(native.lib().msceer_cnn_predict(net.ctx.handle, net._h, ctypes.c_void_p(d.addr), shape[2], shape[1],
                                                 shape[0], ctypes.c_void_p(d.addr), native.DEVICE_PTRS), "predict")
    assert np.array_equal(d.download(np.uint32, f.size), got.ravel().view(np.uint32))


@pytest.mark.parametrize("shape", [(1, 1, 33), (2, 15, 31), (8, 17, 33), (9, 4, 64), (33, 5, 3)])
def test_gradient(net, shape):
    print("cnn tiles gradient", shape, flush=True)
    f, p = _values(shape), _params(35)
    t = (synth.Stream(42).uniform(f.size).reshape(shape) < 0.3).astype(np.uint8)
    net.set_params(p)
    loss, g = net.gradient(f, t, pos_weight=2.0)
    lref, gref = oracle_lib.cnn_gradient(p, f, t, 2.0, quant=1)
    assert abs(loss - lref) < 1e-4 * max(1.0, lref)
    rel = float(np.linalg.norm(g.astype(np.float64) - gref) / np.linalg.norm(gref))
    print(f"  relative error {rel:.2e}", flush=True)
    assert rel < 3e-2
