"""Loop kernels that read inputs through transposes, slices, broadcasts,
reshapes and concatenations: one vector load per input where a thread's
elements stay consecutive, element reads elsewhere. The same values, bit for
bit, as numpy's, at sizes on both sides of that line."""
import numpy as np
import pytest

from pjrtx_amd.hlo import Builder

pytestmark = pytest.mark.gpu

NP = {"f32": np.float32, "f16": np.float16, "s8": np.int8, "s32": np.int32, "s64": np.int64}


def _draw(shape, dt, seed, most):
    return np.random.default_rng(seed).integers(-most, most, shape).astype(NP[dt])


def _check(client, dt, shapes, make, want, most=100):
    args = [_draw(s, dt, i, most) for i, s in enumerate(shapes)]
    b = Builder()
    exe = client.compile(b.build(make(b, [b.param(s, dt) for s in shapes])))
    for got, ref in zip(exe(*args, dtypes=[dt] * len(args)), want(*args)):
        np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("dt", list(NP))
@pytest.mark.parametrize("inner", [1, 3, 4, 6, 8, 12, 16, 24, 130, 256])
def test_transpose_broadcast_reshape(client, dt, inner):
    m, h = 10, 6

    def make(b, p):
        x, row, tab = p
        t = b.transpose(x, [1, 0, 2])                                     # [h, m, inner]
        s = b.add(t, b.broadcast_in_dim(row, (h, m, inner), [2]))
        s = b.add(s, b.broadcast_in_dim(tab, (h, m, inner), [1, 2]))
        return [s, b.add(b.reshape(t, (h * m * inner,)), b.reshape(s, (h * m * inner,)))]

    def want(x, row, tab):
        s = x.transpose(1, 0, 2) + row + tab
        return [s, (x.transpose(1, 0, 2) + s).reshape(-1)]

    _check(client, dt, [(m, h, inner), (inner,), (m, inner)], make, want)


@pytest.mark.parametrize("dt", ["f32", "f16", "s8"])
@pytest.mark.parametrize("inner,lo,hi", [(32, 8, 24), (32, 0, 16), (32, 16, 32), (32, 4, 20), (32, 3, 19), (48, 16, 40), (20, 4, 12)])
def test_slices(client, dt, inner, lo, hi):
    def make(b, p):
        s = b.slice(p[0], [1, lo], [9, hi])
        return [b.add(s, p[1]), b.add(b.slice(p[0], [0, 0], [8, inner], [1, 2]) if inner // 2 == hi - lo else s, p[1])]

    def want(x, y):
        return [x[1:9, lo:hi] + y, (x[0:8, ::2] if inner // 2 == hi - lo else x[1:9, lo:hi]) + y]

    _check(client, dt, [(9, inner), (8, hi - lo)], make, want)


@pytest.mark.parametrize("dt", ["f32", "f16", "s8"])
@pytest.mark.parametrize("sizes", [(64, 64), (8, 24, 16), (16, 8, 8), (4, 12), (5, 11), (16, 16, 1, 15), (2, 6, 24), (32, 0, 32)])
@pytest.mark.parametrize("dim", [0, 1])
def test_concatenations(client, dt, sizes, dim):
    sizes = [s for s in sizes if s] if dim == 0 else list(sizes)
    shapes = [(s, 40) if dim == 0 else (5, s) for s in sizes]
    total = (sum(sizes), 40) if dim == 0 else (5, sum(sizes))

    def make(b, p):
        return [b.add(b.concatenate(p[:-1], dim), p[-1])]

    def want(*a):
        return [np.concatenate(a[:-1], dim) + a[-1]]

    _check(client, dt, shapes + [total], make, want)


@pytest.mark.parametrize("dt", ["f32", "f16"])
@pytest.mark.parametrize("heads,rows,d", [(4, 9, 128), (3, 5, 64), (2, 7, 24), (2, 3, 12), (1, 4, 2)])
def test_rotary_halves(client, dt, heads, rows, d):
    """x cos + concat(-x2, x1) sin, transposed to heads: both halves of a row."""
    def make(b, p):
        x, cos, sin = p
        t = b.transpose(x, [1, 0, 2])
        rot = b.concatenate([b.negate(b.slice(t, [0, 0, d // 2], [heads, rows, d])),
                             b.slice(t, [0, 0, 0], [heads, rows, d // 2])], 2)
        tab = lambda v: b.broadcast_in_dim(b.concatenate([v, v], 1), (heads, rows, d), [1, 2])  # noqa: E731
        return [b.add(b.multiply(t, tab(cos)), b.multiply(rot, tab(sin)))]

    def want(x, cos, sin):
        t = x.transpose(1, 0, 2)
        rot = np.concatenate([-t[..., d // 2:], t[..., :d // 2]], -1)
        return [t * np.concatenate([cos, cos], 1) + rot * np.concatenate([sin, sin], 1)]

    args = [(rows, heads, d), (rows, d // 2), (rows, d // 2)]
    # Sums of two products of integers up to 31 stay below 2^11: exact in f16
    # whether or not the product is rounded before the sum (a contracted
    # multiply-add does not).
    _check(client, dt, args, make, want, most=31)
