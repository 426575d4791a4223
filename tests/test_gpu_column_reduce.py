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
          ((70, 33, 6), (0,)), ((33, 70, 514), (1,)), ((16, 9, 12, 20), (0, 2)), ((40, 50, 24), (0, 1)), ((65, 0), (0,)),
          ((64, 1), (0,)), ((200, 16), (0,)), ((3, 256, 2), (1,)), ((1024, 3), (0,)), ((1025, 2), (0,))]


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


# 256 lanes (odd rows of 16,129 outputs and more), a last block of one output,
# splits; serial threads beside the bounds of their rule.
WIDE = [((256, 16385), (0,)), ((1000, 16129), (0,)), ((300, 40001), (0,)), ((2, 257, 16385), (1,)),
        ((64, 57343), (0,)), ((64, 57345), (0,)), ((256, 57348), (0,))]


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape,dims", WIDE)
def test_wide_rows(client, shape, dims, dt):
    """Whole numbers, whose sums are exact in any order in f32 (and so after
    the one rounding of a 16-bit result)."""
    x = np.random.default_rng(shape[-1]).integers(-8, 9, shape)
    bits = to_bf16_bits(x.astype(np.float32)) if dt == "bf16" else x.astype(np.float16 if dt == "f16" else np.float32)
    b = Builder()
    p = b.param(shape, dt)
    got = client.compile(b.build([b.sum(p, list(dims)), *b.argmax(p, dims[0], "s32")]))(bits, dtypes=[dt])
    vals = [from_bf16_bits(g) if dt == "bf16" else np.asarray(g, np.float32) for g in got[:2]]
    want = x.sum(axis=dims).astype(np.float32)
    if dt != "f32":
        want = from_bf16_bits(to_bf16_bits(want)) if dt == "bf16" else want.astype(np.float16).astype(np.float32)
    np.testing.assert_array_equal(vals[0], want)
    np.testing.assert_array_equal(vals[1], x.max(axis=dims).astype(np.float32))
    np.testing.assert_array_equal(got[2], np.argmax(x, dims[0]).astype(np.int32))


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("shape", [(33, 40), (300, 520), (1000, 1030)])
def test_f16_sums(client, shape, dt):
    """Lanes that fold f16 values as they are: against the float64 sum, f32
    accumulation (below 1e-6 of the magnitudes' sum) and one rounding."""
    x = np.random.default_rng(shape[0]).standard_normal(shape).astype(np.float32)
    bits = to_bf16_bits(x) if dt == "bf16" else x.astype(np.float16)
    vals = (from_bf16_bits(bits) if dt == "bf16" else bits).astype(np.float64)
    b = Builder()
    p = b.param(shape, dt)
    outs = client.compile(b.build([b.sum(p, [0]), b.sum(b.convert(p, "f32"), [0])]))(bits, dtypes=[dt])
    want, slack = vals.sum(0), 1e-6 * np.abs(vals).sum(0)
    assert (np.abs(outs[1] - want) <= slack).all()
    narrow = from_bf16_bits(outs[0]) if dt == "bf16" else outs[0].astype(np.float64)
    assert (np.abs(narrow - want) <= {"bf16": 2.0 ** -8, "f16": 2.0 ** -11}[dt] * np.abs(want) + slack).all()


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
