"""Reductions over leading or middle dims (the last dim kept): lanes span
outputs, lane rows and splits share the reduced elements."""
import numpy as np
import pytest

from pjrtx_amd.hlo import Builder
from pjrtx_amd.pjrt import from_bf16_bits, to_bf16_bits

pytestmark = pytest.mark.gpu

# Below and at the schedule's threshold (32), one split and many, vectors of
# 8, 4, 2 and 1 elements, lanes past the last output, one output.
SHAPES = [((31, 40), (0,)), ((32, 40), (0,)), ((1000, 5632), (0,)), ((1001, 7), (0,)), ((4099, 1), (0,)),
          ((70, 33, 6), (0,)), ((33, 70, 514), (1,)), ((16, 9, 12, 20), (0, 2)), ((40, 50, 24), (0, 1)), ((65, 0), (0,))]


@pytest.mark.parametrize("dt", ["f32", "bf16", "s32", "f64"])
@pytest.mark.parametrize("shape,dims", SHAPES)
def test_sum_max_min(client, shape, dims, dt):
    rng = np.random.default_rng(len(shape) + shape[0])
    if dt == "s32":
        x = rng.integers(-1000, 1000, shape).astype(np.int32)
    else:
        x = rng.standard_normal(shape).astype(np.float64 if dt == "f64" else np.float32)
    bits = to_bf16_bits(x) if dt == "bf16" else x
    vals = from_bf16_bits(bits) if dt == "bf16" else x
    b = Builder()
    p = b.param(shape, dt)
    init = -2 ** 31 if dt == "s32" else -np.inf
    outs = [b.sum(p, list(dims))]
    if np.prod(shape):
        outs += [b.reduce(p, b.constant(init, dt), list(dims), "maximum")]
    got = client.compile(b.build(outs))(bits, dtypes=[dt])
    n = int(np.prod([shape[d] for d in dims]))
    want = vals.astype(np.float64).sum(axis=dims)
    if dt == "s32":
        np.testing.assert_array_equal(got[0], want.astype(np.int64).astype(np.int32))
    elif dt == "bf16":
        # f32 sum (error below 1e-6 of the magnitudes' sum), one bf16 rounding.
        assert (np.abs(from_bf16_bits(got[0]) - want) <= 2.0 ** -8 * np.abs(want) + 1e-6 * n).all()
    else:
        eps = 2.0 ** -52 if dt == "f64" else 2.0 ** -23
        assert (np.abs(got[0] - want) <= eps * n * (1 + np.abs(vals).max(initial=0))).all()
    if len(got) > 1:
        m = from_bf16_bits(got[1]) if dt == "bf16" else got[1]
        np.testing.assert_array_equal(m, vals.max(axis=dims).astype(m.dtype))


@pytest.mark.parametrize("rows,cols", [(33, 8), (1000, 96), (4099, 1030), (40, 1)])
def test_argmax_over_rows(client, rows, cols):
    """First maximum per column across lane rows and splits, NaN first."""
    rng = np.random.default_rng(rows)
    x = rng.integers(0, 12, (rows, cols)).astype(np.float32)
    x[rows // 2, 0] = np.nan
    x[rows - 1, 0] = np.nan
    b = Builder()
    v, i = b.argmax(b.param((rows, cols), "f32"), 0, "s32")
    vals, idx = client.compile(b.build([v, i]))(x)
    np.testing.assert_array_equal(idx, np.argmax(x, 0).astype(np.int32))
    np.testing.assert_array_equal(vals, np.take_along_axis(x, np.argmax(x, 0)[None], 0)[0])
