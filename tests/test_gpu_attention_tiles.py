"""attn_pipe's workgroup shapes (32, 64 and 128 queries, one and two key ways)
at both head dims: ragged lengths, grouped heads, cached prefixes, queries
with no allowed key and inputs that are not finite, against the float64
oracle. The bar is test_gpu_attention's: probabilities are rounded to the
input type before the division by their sum."""
import numpy as np
import pytest

from oracle import attention as A
from pjrtx_amd import programs
from test_planner import attention_then_transpose
from test_gpu_attention import assert_close16, from_bits, sdpa_exe, to_bits

pytestmark = pytest.mark.gpu


def _run(client, dt, d, sizes, spoil=None):
    b, sq, hq, skv, hkv, tok = sizes
    rng = np.random.default_rng(sq * 7 + skv + d)
    qs, kvs = (b, sq, hq, d), (b, skv, hkv, d)
    q, k, v = (to_bits(rng.standard_normal(s), dt) for s in (qs, kvs, kvs))
    if spoil:
        spoil(q, k, v)
    (out,) = sdpa_exe(client, dt, qs, kvs)(q, k, v, np.array(tok, np.int32), dtypes=[dt, dt, dt, None])
    with np.errstate(invalid="ignore"):
        want = A.sdpa_f64(from_bits(q, dt), from_bits(k, dt), from_bits(v, dt), np.int32(tok))
    return from_bits(out, dt), want, out, v


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sizes", [
    (1, 17, 1, 17, 1, 0),        # 32 queries, two key ways
    (1, 200, 8, 333, 2, 100),
    (2, 64, 3, 700, 3, 636),
    (1, 32, 4, 64, 4, 32),       # the second way's only block is masked for most queries
    (4, 300, 16, 300, 4, 0),     # 64 queries
    (4, 330, 15, 470, 5, 139),   # batch * heads not a multiple of 8
    (8, 140, 48, 140, 6, 0),     # 128 queries
    (7, 130, 53, 195, 53, 64),
])
def test_workgroup_shapes(client, dt, d, sizes):
    got, want, out, v = _run(client, dt, d, sizes)
    assert_close16(got, want)
    b, sq, hq, skv, hkv, tok = sizes
    if tok == 0:  # query 0 sees key 0 alone: its value row exactly
        np.testing.assert_array_equal(np.asarray(out)[:, 0], np.repeat(np.asarray(v)[:, 0], hq // hkv, axis=1))


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sizes", [(1, 17, 1, 17, 1, 0), (2, 64, 3, 700, 3, 636), (4, 330, 15, 470, 5, 139), (1, 256, 8, 256, 8, 0)])
def test_register_staged_tiles(client, dt, d, sizes, monkeypatch):
    """attn_tiles, which takes heads whose keys or values span 2 GiB."""
    monkeypatch.setenv("PJRTX_ATTN_PIPE", "0")
    got, want, _, _ = _run(client, dt, d, sizes)
    assert_close16(got, want)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sizes", [(1, 40, 2, 150, 1, -3), (4, 300, 16, 300, 4, -1), (8, 140, 48, 140, 48, -2)])
def test_queries_with_no_allowed_key(client, d, sizes):
    got, want, _, _ = _run(client, "bf16", d, sizes)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    assert np.isnan(want).any()
    assert_close16(np.nan_to_num(got), np.nan_to_num(want))


@pytest.mark.parametrize("sizes", [(1, 96, 4, 200, 4, 104), (4, 300, 16, 300, 16, 0), (8, 140, 48, 140, 48, 0)])
def test_values_that_are_not_finite(client, sizes):
    """An infinite value passes through (a quotient's special case), a NaN key
    poisons the queries that may see it and no other."""
    def spoil(q, k, v):
        v[0, 0, 0, 5] = 0x7f80
        k[0, 70, 1, 3] = 0x7fc0
    got, want, _, _ = _run(client, "bf16", 128, sizes, spoil)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
    assert np.isposinf(want).any() and np.isnan(want).any()
    keep = np.isfinite(want)
    assert_close16(np.where(keep, got, 0), np.where(keep, want, 0))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bh", [(1, 3), (4, 72)])        # 32 queries and two key ways, 128 queries
@pytest.mark.parametrize("blocks", [(0,), (0, 1), (2,), (0, 1, 2, 3)])
def test_f16_scores_that_overflow(client, d, bh, blocks):
    """Key blocks of 64 whose f16 scores all round to -inf weigh nothing, also
    before any other block was seen; a row of nothing else is NaN."""
    b, h = bh
    s = 256
    rng = np.random.default_rng(d)
    q, k, v = (rng.standard_normal((b, h, s, d)).astype(np.float32) for _ in range(3))
    q = np.abs(q) / d ** 0.5 + 16
    k /= 64
    for blk in blocks:
        k[:, :, 64 * blk:64 * blk + 64] = -66000 / (16 * d) - 8  # a score of -66000 and below
    args = [to_bits(x, "f16") for x in (q, k, v)]
    (out,) = client.compile(programs.c3_attention(b, h, s, d, False, dtype="f16"))(*args, dtypes=["f16"] * 3)
    with np.errstate(invalid="ignore"):
        want = A.attention_graph_ref(*(from_bits(x, "f16") for x in args), "f16")
    got = from_bits(out, "f16")
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    assert np.isnan(want).all() == (len(blocks) == 4)
    assert_close16(np.nan_to_num(got), np.nan_to_num(want))


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape", [(1, 16, 100, 128), (3, 5, 33, 64), (2, 3, 17, 40), (2, 130, 160, 128)])
def test_result_written_transposed(client, shape, dt):
    rng = np.random.default_rng(shape[2])
    args = [rng.standard_normal(shape).astype(np.float32) for _ in range(3)]
    args = args if dt == "f32" else [to_bits(a, dt) for a in args]
    (plain,) = client.compile(programs.c3_attention(*shape, True, dtype=dt))(*args, dtypes=[dt] * 3)
    (got,) = client.compile(attention_then_transpose(shape, [0, 2, 1, 3], dt))(*args, dtypes=[dt] * 3)
    np.testing.assert_array_equal(np.asarray(got).view(np.uint8), np.ascontiguousarray(np.asarray(plain).transpose(0, 2, 1, 3)).view(np.uint8))
