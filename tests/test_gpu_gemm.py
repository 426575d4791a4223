"""dot_general's MFMA block tiles (kernels/gemm.hip): every tile in every
operand layout at ragged sizes, k-splits, and operands that need padded rows,
against the float64 product."""
import numpy as np
import pytest

from oracle import ops
from pjrtx_amd.hlo import Builder
from pjrtx_amd.pjrt import from_bf16_bits, to_bf16_bits

pytestmark = pytest.mark.gpu


def _dot(client, spec, sizes, dt="bf16", out_dt=None, seed=0):
    """dot_general of the spec (batch b, free m and n, contracted k, in any
    order) and the float64 product of the same values."""
    ls, rs = spec.split(",")
    rng = np.random.default_rng(seed)
    arrs = []
    for dims in (ls, rs):
        v = rng.standard_normal([sizes[c] for c in dims]).astype(np.float32)
        arrs.append(to_bf16_bits(v) if dt == "bf16" else v.astype(np.float16))
    vals = [from_bf16_bits(a) if dt == "bf16" else a.astype(np.float32) for a in arrs]
    batch = (tuple(i for i, c in enumerate(ls) if c == "b"), tuple(i for i, c in enumerate(rs) if c == "b"))
    contract = ((ls.index("k"),), (rs.index("k"),))
    b = Builder()
    x, y = (b.param(a.shape, dt) for a in arrs)
    exe = client.compile(b.build([b.dot_general(x, y, batch=batch, contract=contract, out_dtype=out_dt)]))
    (got,) = exe(*arrs, dtypes=[dt, dt])
    got = from_bf16_bits(got) if dt == "bf16" and out_dt is None else got.astype(np.float32)
    return got, ops.dot_general_f64(vals[0], vals[1], batch[0], batch[1], contract[0], contract[1])


def _check(got, want, k, dt, out_dt):
    # f32 sums of k products of N(0,1) values in any order: error of at most
    # about k 2^-24 of the sum of magnitudes (0.64 k), far below; then one
    # rounding to the result type.
    ulp = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11}[dt] if out_dt is None else 0.0
    tol = ulp * np.abs(want) + 1e-6 * k ** 0.5 * 4
    assert got.shape == want.shape
    assert (np.abs(got - want) <= tol).all(), np.abs(got - want).max()


TILES = [0, 1, 2, 3, 4, 5]
LAYOUTS = ["mk,kn", "mk,nk", "km,kn", "km,nk"]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("spec", LAYOUTS)
def test_tiles_and_layouts(client, tile, spec, monkeypatch):
    """Whole tiles, ragged edges in m, n and k, one k-tile and many, and a
    product smaller than the tile."""
    monkeypatch.setenv("PJRTX_GEMM_TILE", str(tile))
    for i, (m, n, k) in enumerate([(256, 256, 64), (264, 520, 136), (40, 72, 1096), (16, 8, 8), (520, 264, 200)]):
        got, want = _dot(client, spec, {"m": m, "n": n, "k": k}, seed=i)
        _check(got, want, k, "bf16", None)


@pytest.mark.parametrize("dt,out_dt", [("f16", None), ("bf16", "f32"), ("f16", "f32")])
@pytest.mark.parametrize("tile", TILES)
def test_tile_types(client, tile, dt, out_dt, monkeypatch):
    monkeypatch.setenv("PJRTX_GEMM_TILE", str(tile))
    for spec in ("bmk,bkn", "bkm,bnk"):
        got, want = _dot(client, spec, {"b": 3, "m": 72, "n": 264, "k": 328}, dt, out_dt, seed=tile)
        _check(got, want, 328, dt, out_dt)


@pytest.mark.parametrize("m,n,k", [(17, 33, 4099), (64, 128, 8192), (9, 2048, 2040), (33, 1000, 3001), (128, 64, 20000)])
def test_k_splits(client, m, n, k):
    """Few tiles and a long k: the plan splits k and sums f32 partials."""
    for spec in LAYOUTS:
        got, want = _dot(client, spec, {"m": m, "n": n, "k": k}, seed=m)
        _check(got, want, k, "bf16", None)


@pytest.mark.parametrize("sizes", [(2, 19, 21, 13), (3, 65, 130, 67), (1, 100, 9, 1), (2, 1, 40, 70), (2, 40, 1, 70),
                                   (2, 5, 24, 64), (1, 8, 23, 65), (2, 19, 21, 61), (1, 100, 9, 57)])
def test_dimension_orders(client, sizes):
    """Every order of the operands' dimensions, odd sizes (rows that are not
    16-byte aligned are padded first), unit dimensions, decode rows."""
    size = dict(zip("bmnk", sizes))
    for lhs in ("bmk", "bkm", "mbk", "kbm", "mkb"):
        for rhs in ("bkn", "bnk", "kbn", "nbk", "knb"):
            got, want = _dot(client, f"{lhs},{rhs}", size, seed=size["k"])
            _check(got, want, size["k"], "bf16", None)


@pytest.mark.parametrize("lhs,rhs,out,contract", [
    ("akum", "kn", "aumn", ((1,), (0,))),        # u: one element between two free dims that are apart
    ("mk", "akun", "maun", ((1,), (1,))),
    ("mkc", "knuc", "mnu", ((1, 2), (0, 3))),    # between two contracted ones
    ("aumk", "kn", "aumn", ((3,), (0,))),        # between two that follow each other
    ("akm", "kn", "amn", ((1,), (0,))),          # free dims that are apart, contracted ones in another order
    ("mk", "akn", "man", ((1,), (1,))),
    ("akm", "nkc", "amnc", ((1,), (1,))),
    ("mkc", "nck", "mn", ((1, 2), (2, 1))),
    ("kcm", "nkc", "mn", ((1, 0), (2, 1))),
])
@pytest.mark.parametrize("dt", ["bf16", "f32"])
def test_dims_that_do_not_merge(client, lhs, rhs, out, contract, dt):
    size = dict(a=2, c=6, k=40, m=12, n=24, u=1)
    vals = [np.random.default_rng(i).integers(-3, 4, [size[c] for c in s]).astype(np.float32) for i, s in enumerate((lhs, rhs))]
    b = Builder()
    x, y = (b.param(v.shape, dt) for v in vals)
    exe = client.compile(b.build([b.dot_general(x, y, contract=contract, out_dtype="f32")]))
    (got,) = exe(*(to_bf16_bits(v) if dt == "bf16" else v for v in vals), dtypes=[dt] * 2)
    # Whole numbers: every sum is exact in f32.
    np.testing.assert_array_equal(got, np.einsum(f"{lhs},{rhs}->{out}", *vals))


def test_ragged_rows_of_many_batches(client):
    """More batches than a launch's grid holds of padded rows."""
    b, m, k, n = 65541, 9, 16, 12
    rng = np.random.default_rng(1)
    x, y = (rng.integers(-3, 4, s).astype(np.float32) for s in ((b, m, k), (b, k, n)))
    h = Builder()
    d = h.dot_general(h.param(x.shape, "bf16"), h.param(y.shape, "bf16"), batch=((0,), (0,)), contract=((2,), (1,)),
                      out_dtype="f32")
    (got,) = client.compile(h.build([d]))(to_bf16_bits(x), to_bf16_bits(y), dtypes=["bf16"] * 2)
    np.testing.assert_array_equal(got, np.matmul(x, y))


@pytest.mark.parametrize("spec,dt,out_dt", [("mk,kn", "bf16", "f32"), ("mk,nk", "bf16", "f32"), ("mk,kn", "f16", "f32"),
                                            ("mk,nk", "f16", "f32"), ("mk,nk", "bf16", "bf16"), ("mk,kn", "bf16", "bf16")])
def test_rows_of_four_million_elements(client, spec, dt, out_dt):
    """Rows past the block tiles' 32-bit offsets go to mfma_gemm; a ragged
    last k-tile. Whole numbers whose partial sums (a random walk, deviation
    8,200) stay far below 2^24: every f32 sum is exact."""
    m, n, k = 9, 16, (1 << 22) + 72
    rng = np.random.default_rng(5)
    x, y = (rng.integers(-2, 3, s).astype(np.float32) for s in ((m, k), (k, n) if spec == "mk,kn" else (n, k)))
    b = Builder()
    contract = ((1,), (0,) if spec == "mk,kn" else (1,))
    dot = b.dot_general(b.param(x.shape, dt), b.param(y.shape, dt), contract=contract, out_dtype=out_dt)
    store = to_bf16_bits if dt == "bf16" else (lambda v: v.astype(np.float16))
    (got,) = client.compile(b.build([dot]))(store(x), store(y), dtypes=[dt] * 2)
    want = x @ (y if spec == "mk,kn" else y.T)
    np.testing.assert_array_equal(got, want if out_dt == "f32" else to_bf16_bits(want))


@pytest.mark.parametrize("m", [1, 3, 4])
@pytest.mark.parametrize("n,k", [(9, 512), (33, 2048), (257, 1032), (511, 520)])
def test_decode_rows_of_few_ragged_columns(client, m, n, k):
    for spec in LAYOUTS:
        for dt, out_dt in (("bf16", None), ("f16", "f32")):
            got, want = _dot(client, spec, {"m": m, "n": n, "k": k}, dt, out_dt, seed=n)
            _check(got, want, k, dt, out_dt)


@pytest.mark.parametrize("sizes", [(1, 2, 16, 58), (1, 6, 512, 44), (3, 7, 896, 73), (1, 8, 40, 127), (2, 5, 33, 129)])
def test_decode_rows_of_a_short_ragged_contraction(client, sizes):
    size = dict(zip("bmnk", sizes))
    for spec in ("bmk,bkn", "bmk,bnk", "bkm,bkn", "bkm,bnk"):
        for dt, out_dt in (("bf16", None), ("f16", "f32")):
            got, want = _dot(client, spec, size, dt, out_dt, seed=size["k"])
            _check(got, want, size["k"], dt, out_dt)


def test_same_bits_on_every_call(client):
    sizes = {"m": 100, "n": 520, "k": 4104}
    a, _ = _dot(client, "mk,kn", sizes)
    b, _ = _dot(client, "mk,kn", sizes)
    np.testing.assert_array_equal(a, b)
