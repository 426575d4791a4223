"""Edges of the sort kernels' paths: wave and workgroup merge rounds, rows of
one LDS block and several runs, unaligned rows, positions folded out of the
operands, and top-k chunks with many equal keys. Bit-exact (oracle/sort.py)."""
import numpy as np
import pytest

from oracle import sort as S
from pjrtx_amd.hlo import Builder
from pjrtx_amd.pjrt import DeviceArray, to_bf16_bits

pytestmark = pytest.mark.gpu


def _keys(rng, shape, dt, distinct):
    x = rng.integers(-distinct, distinct, shape) if distinct else rng.standard_normal(shape)
    if dt == "s32":
        return (x if distinct else x * 4e8).astype(np.int32)
    x = x.astype(np.float32)
    return to_bf16_bits(x) if dt == "bf16" else x


def _same(got, want):
    np.testing.assert_array_equal(np.asarray(got).view(np.uint8), np.ascontiguousarray(want).view(np.uint8))


def _argsort(client, x, dt, dim, direction="LT", index="s32"):
    b = Builder("jit_argsort")
    p = b.param(x.shape, dt)
    v, i = b.sort([p, b.iota(x.shape, dim, index)], dim, direction)
    return client.compile(b.build([v, i]))(x, dtypes=[dt])


@pytest.mark.parametrize("dt", ["f32", "bf16", "s32"])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 511, 512, 513, 1024, 1025, 8191, 8192, 8193, 16384, 16385, 40003, 65536])
def test_argsort_lengths(client, n, dt):
    rng = np.random.default_rng(n)
    for distinct in (0, 3):
        x = _keys(rng, (3, n), dt, distinct)
        pos = np.broadcast_to(np.arange(n, dtype=np.int32), x.shape).copy()
        ct = "SIGNED" if dt == "s32" else "TOTALORDER"
        for direction in ("LT", "GT"):
            v, i = _argsort(client, x, dt, 1, direction)
            wv, wi = S.sort_stablehlo([x, pos], 1, ct, direction == "GT", bf16=dt == "bf16")
            _same(v, wv)
            _same(i, wi)


@pytest.mark.parametrize("index,np_index", [("s8", np.int8), ("u16", np.uint16), ("s64", np.int64)])
def test_position_types(client, index, np_index):
    """Positions in the iota's own type, wrapped to its width as the iota is."""
    x = np.random.default_rng(2).standard_normal((2, 9000)).astype(np.float32)
    v, i = _argsort(client, x, "f32", 1, index=index)
    order = np.argsort(x, 1, kind="stable")
    _same(i, order.astype(np_index))
    _same(v, np.take_along_axis(x, order, 1))


@pytest.mark.parametrize("shape,dim", [((9001, 3), 0), ((2, 600, 5), 1), ((20, 4), 0)])
def test_argsort_other_dims(client, shape, dim):
    x = _keys(np.random.default_rng(1), shape, "f32", 50)
    v, i = _argsort(client, x, "f32", dim)
    order = np.argsort(x, dim, kind="stable")
    _same(v, np.take_along_axis(x, order, dim))
    _same(i, order.astype(np.int32))


@pytest.mark.parametrize("rows,n,k", [(1, 300, 256), (3, 2048, 1), (3, 2049, 256), (64, 8192, 50), (5, 8193, 50),
                                      (2, 100000, 256), (1, 1000000, 200), (3, 9000, 257), (3, 50000, 4096),
                                      (3, 50000, 4097), (300, 2050, 5), (3, 8192, 256), (7, 5000, 200),
                                      (5, 9, 8), (5, 8, 1), (300, 512, 8), (3, 511, 9), (3, 513, 8), (3, 65, 7),
                                      (3, 512, 511), (3, 2048, 129), (3, 2049, 129),
                                      (9, 576, 20), (9, 576, 40), (9, 1024, 41), (5, 1032, 41), (5, 1032, 100)])
@pytest.mark.parametrize("distinct", [0, 2, 40])
def test_top_k_edges(client, rows, n, k, distinct):
    """Chunks of one, two and four groups a thread, one to three rounds, and
    the block and merge paths above k = 256; with 2 * `distinct` different keys
    whole chunks tie with the threshold."""
    rng = np.random.default_rng(n + k)
    for dt in ("bf16", "f32"):
        x = _keys(rng, (rows, n), dt, distinct)
        b = Builder("jit_topk")
        v, i = b.top_k(b.param((rows, n), dt), k)
        vals, idx = client.compile(b.build([v, i]))(x, dtypes=[dt])
        wv, wi = S.top_k(x, k, bf16=dt == "bf16")
        _same(idx, wi)
        _same(vals, wv)


@pytest.mark.parametrize("order", ["random", "ascending", "descending", "equal"])
@pytest.mark.parametrize("dt", ["bf16", "f32"])
def test_top_k_as_many_as_threads(client, dt, order):
    """k = 256, where the threads' least words bound little and sorted lists
    give every thread words of like rank: the results, and that few words are
    ranked (by counting, quadratic: 18 times k = 50's time and more when every
    word was; at most 5 times since)."""
    def run(rows, n, k):
        x = np.random.default_rng(n).standard_normal((rows, n)).astype(np.float32)
        x = {"random": x, "ascending": np.sort(x, 1), "descending": -np.sort(x, 1), "equal": np.ones_like(x)}[order]
        x = to_bf16_bits(x) if dt == "bf16" else x
        b = Builder("jit_topk")
        exe = client.compile(b.build(list(b.top_k(b.param(x.shape, dt), k))))
        args = [client.buffer(x, dt)]
        vals, idx = (o.to_numpy() for o in exe.execute_buffers(args))
        wv, wi = S.top_k(x, k, bf16=dt == "bf16")
        _same(idx, wi)
        _same(vals, wv)
        exe.run_loop(args, 3)
        return min(exe.run_loop(args, 10) for _ in range(5))

    for rows, n in ((17, 54716), (64, 8192)):
        assert run(rows, n, 256) < 12 * run(rows, n, 50)


def test_short_rows_take_less(client):
    """Rows are merged only as far as they go, short ones are not bounded first
    (each took about as long as the longest a wave holds: 15 and 44 us where 5 and 10
    are taken now), and a bound has groups of words to rank (56 and 28). 4096 rows, so that
    the GPU's time counts."""
    def best(n, k, dt="f32"):
        b = Builder("jit_short")
        p = b.param((4096, n), dt)
        exe = client.compile(b.build(list(b.top_k(p, k) if k else b.sort([p, b.iota((4096, n), 1)], 1))))
        args = [client.buffer(_keys(np.random.default_rng(n), (4096, n), dt, 0), dt)]
        exe.run_loop(args, 10)
        return min(exe.run_loop(args, 30) for _ in range(5))

    assert best(8, 0) < 0.6 * best(512, 0)
    assert best(64, 20) < 0.7 * best(2000, 20)
    assert best(576, 20, "bf16") < 1.7 * best(2048, 20, "bf16")


def test_sort_in_a_fixed_block(client, plugin):
    """A row whose two merge buffers exceed the allocation-free block's 64 MiB
    is sorted by the one-buffer network there."""
    n = 1 << 22
    x = np.random.default_rng(0).integers(-2 ** 31, 2 ** 31 - 1, n).astype(np.int32)
    b = Builder("jit_sort")
    (v,) = b.sort([b.param((n,), "s32")], 0)
    exe = client.compile(b.build([v]))
    src, dst = DeviceArray.from_numpy(plugin, x), DeviceArray(plugin, x.nbytes)
    used = exe.execute_noalloc([src.ptr], [dst.ptr])
    plugin.hip_check(plugin.lib.pjrtx_hip_synchronize(0))
    np.testing.assert_array_equal(dst.to_numpy(np.int32, (n,)), np.sort(x))
    assert used < 64 << 20
    src.free()
    dst.free()
