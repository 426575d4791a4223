"""Block-tile products that do more than multiply: a residual or bias row added
in the epilogue, members of one launch, and a product written transposed,
against the float64 result."""
import json

import numpy as np
import pytest

from oracle import ops
from pjrtx_amd.hlo import Builder

pytestmark = pytest.mark.gpu


def _draw(shape, dt, seed):
    v = np.random.default_rng(seed).standard_normal(shape).astype(np.float32)
    bits = ops.f32_to_bf16_bits(v) if dt == "bf16" else v.astype(np.float16)
    return bits, _f64(bits, dt)


def _f64(a, dt):
    return (ops.bf16_bits_to_f32(a) if dt == "bf16" else np.asarray(a, np.float32)).astype(np.float64)


ULP = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11}


def _steps(exe):
    return json.loads(exe.optimized_program())["steps"]


def _check_sum(got, prod, x, k, dt):
    # The product is rounded to the type, then the sum (half an ulp each, of at
    # most twice the value's power of two); f32 sums add far less (1e-6 sqrt(k)).
    tol = ULP[dt] * (np.abs(prod) + np.abs(prod + x)) + 4e-6 * k ** 0.5
    assert (np.abs(_f64(got, dt) - (prod + x)) <= tol).all()


SIZES = [(9, 16, 64), (256, 256, 128), (129, 1000, 72), (40, 264, 8200), (33, 37, 4099), (300, 513, 65)]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("add", ["row", "full", "left"])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_added_row_and_residual(client, m, n, k, add, dt):
    """Whole and ragged tiles, split k, rows that are not 16-byte aligned."""
    (a, av), (w, wv) = _draw((m, k), dt, 1), _draw((k, n), dt, 2)
    x, xv = _draw((n,) if add == "row" else (m, n), dt, 3)
    b = Builder()
    pa, pw, px = b.param((m, k), dt), b.param((k, n), dt), b.param(x.shape, dt)
    y = b.dot_general(pa, pw, contract=((1,), (0,)))
    z = b.add(px, y) if add == "left" else b.add(y, b.broadcast_in_dim(px, (m, n), [1]) if add == "row" else px)
    exe = client.compile(b.build([z]))
    assert len(_steps(exe)) == 1
    (got,) = exe(a, w, x, dtypes=[dt] * 3)
    _check_sum(got, av @ wv, xv, k, dt)


# Right operands with no, two and three free dims; batched; contracted last.
# 72 elements are summed in one launch of the block tiles, 8200 in k-splits.
FREE_DIMS = [("mk", "k", "m"), ("mk", "kgh", "mgh"), ("mk", "ghk", "mgh"), ("km", "kgh", "mgh"), ("mk", "kfgh", "mfgh"),
             ("amk", "kgh", "amgh"), ("mk", "gkh", "mgh"), ("akm", "kgh", "amgh"), ("bmk", "bk", "bm"), ("bmk", "bkgh", "bmgh"), ("bkm", "bghk", "bmgh")]


@pytest.mark.parametrize("k", [72, 8200])
@pytest.mark.parametrize("lhs,rhs,out", FREE_DIMS)
@pytest.mark.parametrize("g,h", [(4, 32), (3, 7)])
def test_residual_of_any_free_dims(client, lhs, rhs, out, g, h, k):
    size = dict(a=2, b=3, f=2, g=g, h=h, k=k, m=130)
    shape = lambda s: tuple(size[c] for c in s)  # noqa: E731
    (a, av), (w, wv), (x, xv) = (_draw(shape(s), "bf16", i) for i, s in enumerate((lhs, rhs, out)))
    b = Builder()
    pa, pw, px = (b.param(shape(s), "bf16") for s in (lhs, rhs, out))
    y = b.dot_general(pa, pw, batch=((0,), (0,)) if "b" in lhs else ((), ()),
                      contract=((lhs.index("k"),), (rhs.index("k"),)))
    exe = client.compile(b.build([b.add(px, y)]))
    assert len(_steps(exe)) == 1
    (got,) = exe(a, w, x, dtypes=["bf16"] * 3)
    _check_sum(got, np.einsum(f"{lhs},{rhs}->{out}", av, wv), xv, k, "bf16")


def test_batched_residual_and_bias(client):
    (a, av), (w, wv) = _draw((3, 40, 72), "bf16", 1), _draw((3, 72, 50), "bf16", 2)
    for shape in ((3, 40, 50), (50,)):
        x, xv = _draw(shape, "bf16", 3)
        b = Builder()
        pa, pw, px = b.param((3, 40, 72), "bf16"), b.param((3, 72, 50), "bf16"), b.param(shape, "bf16")
        y = b.dot_general(pa, pw, batch=((0,), (0,)), contract=((2,), (1,)))
        exe = client.compile(b.build([b.add(y, px if len(shape) == 3 else b.broadcast_in_dim(px, (3, 40, 50), [2]))]))
        (got,) = exe(a, w, x, dtypes=["bf16"] * 3)
        _check_sum(got, av @ wv, xv, 72, "bf16")


@pytest.mark.parametrize("m,k,ns", [
    (512, 256, (2048, 256, 256)),   # q/k/v with grouped-query widths
    (9, 4096, (520, 520)),
    (65, 136, (8, 1000, 72, 264)),
    (33, 67, (24, 31)),             # rows of x and of a member are not aligned
])
def test_members_of_one_launch(client, m, k, ns):
    x, xv = _draw((m, k), "bf16", 1)
    ws = [_draw((k, n), "bf16", 2 + i) for i, n in enumerate(ns)]
    b = Builder()
    px = b.param((m, k), "bf16")
    exe = client.compile(b.build([b.dot_general(px, b.param((k, n), "bf16"), contract=((1,), (0,))) for n in ns]))
    assert [s.get("library") for s in _steps(exe)] == ["dot_group"]
    for got, (_, wv) in zip(exe(x, *[w for w, _ in ws], dtypes=["bf16"] * (1 + len(ns))), ws):
        want = xv @ wv
        assert (np.abs(_f64(got, "bf16") - want) <= ULP["bf16"] * np.abs(want) + 4e-6 * k ** 0.5).all()


@pytest.mark.parametrize("batch,lhs,rhs", [("", "mk", "kn"), ("", "km", "kn"), ("", "mk", "nk"), ("b", "bmk", "bkn"), ("b", "bkm", "bnk")])
@pytest.mark.parametrize("dt", ["bf16", "f32"])
def test_transposed_result(client, batch, lhs, rhs, dt):
    for m, n, k in ((72, 264, 136), (9, 17, 33), (8, 40, 24), (300, 129, 4104)):
        size = dict(b=3, m=m, n=n, k=k)
        shapes = [[size[c] for c in s] for s in (lhs, rhs)]
        if dt == "f32":
            vals = [np.random.default_rng(i).standard_normal(s).astype(np.float32) for i, s in enumerate(shapes)]
            pairs = [(v, v.astype(np.float64)) for v in vals]
        else:
            pairs = [_draw(s, dt, i) for i, s in enumerate(shapes)]
        b = Builder()
        x, y = (b.param(s, dt) for s in shapes)
        d = b.dot_general(x, y, batch=((0,), (0,)) if batch else ((), ()), contract=((lhs.index("k"),), (rhs.index("k"),)))
        exe = client.compile(b.build([b.transpose(d, [0, 2, 1] if batch else [1, 0])]))
        assert len(_steps(exe)) == (1 if m > 8 else 2)
        (got,) = exe(*[a for a, _ in pairs], dtypes=[dt] * 2)
        want = np.einsum(f"{lhs},{rhs}->{batch}nm", pairs[0][1], pairs[1][1])
        got = np.asarray(got, np.float64) if dt == "f32" else _f64(got, dt)
        # f32 sums one product at a time: k roundings of half an ulp (2^-24 of
        # the partial sum) add up like a random walk, sqrt(k) of them with 4
        # sigma, and a partial sum of N(0,1) products stays under 5 sqrt(k).
        tol = 20 * k * 2.0 ** -24 if dt == "f32" else ULP[dt] * np.abs(want) + 4e-6 * k ** 0.5
        assert (np.abs(got - want) <= tol).all()


@pytest.mark.parametrize("batch,lhs,rhs", [("", "mk", "kn"), ("", "km", "nk"), ("b", "bmk", "bkn")])
@pytest.mark.parametrize("dt", ["s32", "f32", "f64"])
def test_transposed_result_of_whole_numbers(client, batch, lhs, rhs, dt):
    """The types of the scalar kernel, whose lanes then follow the result's rows."""
    for m, n, k in ((9, 300, 5), (257, 9, 70), (64, 64, 64)):
        size = dict(b=3, m=m, n=n, k=k)
        vals = [np.random.default_rng(i).integers(-9, 10, [size[c] for c in s]) for i, s in enumerate((lhs, rhs))]
        vals = [v.astype({"s32": np.int32, "f32": np.float32, "f64": np.float64}[dt]) for v in vals]
        b = Builder()
        x, y = (b.param(v.shape, dt) for v in vals)
        d = b.dot_general(x, y, batch=((0,), (0,)) if batch else ((), ()), contract=((lhs.index("k"),), (rhs.index("k"),)))
        (got,) = client.compile(b.build([b.transpose(d, [0, 2, 1] if batch else [1, 0])]))(*vals, dtypes=[dt] * 2)
        np.testing.assert_array_equal(got, np.einsum(f"{lhs},{rhs}->{batch}nm", *vals))


@pytest.mark.parametrize("form", ["plain", "f32", "row", "full", "transposed", "members"])
@pytest.mark.parametrize("spec", ["mk,kn", "mk,nk", "km,kn", "km,nk", "akm,kn", "mk,nak"])
def test_small_ragged_products(client, form, spec):
    """Products whose operands would be padded for the tiles, of few enough
    multiplications to go to the scalar kernel in one launch (and, k = 61,
    too many): whole numbers, exact in every form."""
    ls, rs = spec.split(",")
    for dt in ("bf16", "f16"):
        for m, n, k in [(1, 17, 3), (3, 40, 9), (8, 1000, 3), (9, 16, 5), (40, 33, 12), (257, 65, 2), (33, 40, 61)]:
            size = dict(a=3, m=m, n=n, k=k)
            rng = np.random.default_rng(k)
            x, y, y2 = (rng.integers(-3, 4, [size[c] for c in s]).astype(np.float32) for s in (ls, rs, rs))
            store = (lambda v: ops.f32_to_bf16_bits(v)) if dt == "bf16" else (lambda v: v.astype(np.float16))
            b = Builder()
            px, py = b.param(x.shape, dt), b.param(y.shape, dt)
            kw = dict(contract=((ls.index("k"),), (rs.index("k"),)), out_dtype="f32" if form == "f32" else None)
            d = b.dot_general(px, py, **kw)
            lf, rf = ls.replace("k", ""), rs.replace("k", "")
            want = np.einsum(f"{ls},{rs}->{lf}{rf}", x, y)
            args, outs, wants = [x, y], [d], [want]
            if form in ("row", "full"):
                z = rng.integers(-3, 4, want.shape[-1:] if form == "row" else want.shape).astype(np.float32)
                pz = b.param(z.shape, dt)
                outs = [b.add(d, b.broadcast_in_dim(pz, want.shape, [want.ndim - 1]) if form == "row" else pz)]
                args, wants = args + [z], [want + z]
            if form == "transposed":
                perm = list(range(len(lf), want.ndim)) + list(range(len(lf)))
                outs, wants = [b.transpose(d, perm)], [want.transpose(perm)]
            if form == "members":
                outs.append(b.dot_general(px, b.param(y.shape, dt), **kw))
                args, wants = args + [y2], wants + [np.einsum(f"{ls},{rs}->{lf}{rf}", x, y2)]
            got = client.compile(b.build(outs))(*(store(v) for v in args), dtypes=[dt] * len(args))
            for g, w in zip(got, wants):
                # |sums| <= 9 * 61 + 3: beyond 256 bf16 rounds the product and the sum to even numbers.
                if form == "f32":
                    np.testing.assert_array_equal(g, w)
                else:
                    assert (np.abs(_f64(g, dt) - w) <= (0 if np.abs(w).max() < 250 else 2)).all()
