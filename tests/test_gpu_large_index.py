"""Tensors of more than 2^32 elements in generated kernels: the vector loads
and stores take the kernel's 64-bit positions. Made on the GPU (4.3 GB of
bytes), so nothing of that size crosses to the host."""
import numpy as np
import pytest

from pjrtx_amd.hlo import Builder

pytestmark = pytest.mark.gpu

ROWS, COLS = 65537, 65536  # the last row starts at element 2^32


def _reductions():
    b = Builder()
    x = b.param((ROWS, COLS), "s8")
    return b.build([b.reduce(x, b.constant(-128, "s8"), [0], "maximum"),
                    b.reduce(x, b.constant(-128, "s8"), [1], "maximum")])


def test_loop_stores_and_reduction_loads_past_2_32(client):
    b = Builder()
    at = b.iota((ROWS, COLS), 0)
    last = b.compare("EQ", at, b.scalar_like(ROWS - 1, at))
    five, one = (b.broadcast_in_dim(b.constant(v, "s8"), (ROWS, COLS), []) for v in (5, 1))
    (x,) = client.compile(b.build([b.select(last, five, one)])).execute_buffers([])
    over_rows, over_cols = (o.to_numpy() for o in client.compile(_reductions()).execute_buffers([x]))
    np.testing.assert_array_equal(over_rows, np.full(COLS, 5, np.int8))
    np.testing.assert_array_equal(over_cols, np.where(np.arange(ROWS) == ROWS - 1, 5, 1).astype(np.int8))
    # An elementwise kernel that reads it.
    b = Builder()
    p = b.param((ROWS, COLS), "s8")
    (y,) = client.compile(b.build([b.add(p, p)])).execute_buffers([x])
    x.delete()
    over_rows, over_cols = (o.to_numpy() for o in client.compile(_reductions()).execute_buffers([y]))
    np.testing.assert_array_equal(over_rows, np.full(COLS, 10, np.int8))
    np.testing.assert_array_equal(over_cols, np.where(np.arange(ROWS) == ROWS - 1, 10, 2).astype(np.int8))
    y.delete()
