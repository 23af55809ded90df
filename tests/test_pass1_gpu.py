"""Integration of a ramp along x on shapes around the edges of the seed
collection (2048 vertices a work-group, 64 to a row, two strides): every
streamline runs straight along its row to the terminal at its end, so every
label is known exactly -- the row's, and none where the gradient is zero on the
boundary the flow leaves from."""
import numpy as np
import pytest

from msceer_amd import labels, native

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("shape", [(2, 2, 3), (2, 3, 64), (16, 8, 16), (3, 3, 229), (1 + 2 * 5, 7, 131), (33, 31, 67)])
def test_rows_of_a_ramp(ctx, shape, sign):
    print(f"ramp {shape} {sign}", flush=True)
    Z, Y, X = shape
    f = np.broadcast_to(np.arange(X, dtype=np.float32), shape).copy()
    rows = np.arange(Z * Y, dtype=np.int32).reshape(Z, Y, 1)
    end, start = (0, X - 1) if sign < 0 else (X - 1, 0)
    term = np.full(shape, -1, np.int32)
    term[:, :, end] = rows[:, :, 0]
    lab, st = labels.integrate_labels(f, term, sign=sign, ctx=ctx)
    expect = np.broadcast_to(rows, shape).copy()
    expect[:, :, start] = -1
    assert (lab == expect).all(), int((lab != expect).sum())
    assert st["traced_fp32"] + st["over_budget_fp32"] <= Z * Y * (X - 1)
