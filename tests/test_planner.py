"""Host-side tests of the StableHLO importer, the fusion planner and the
kernel generator (no GPU). Structural counterparts of the reference's planner
tests (reference: src/backend/mlx_metal/program_fusion.zig:116-227,
executable_metal_graph_lowering_tests.zig:8-204)."""
import json
import re

import pytest

from pjrtx_amd import programs
from pjrtx_amd.hlo import Builder
from pjrtx_amd.pjrt import PjrtError


def plan(plugin, text):
    return json.loads(plugin.plan_json(text))


def test_c1_is_one_fused_reduction(plugin):
    p = plan(plugin, programs.c1_elementwise_rowsum(64, 256))
    assert len(p["steps"]) == 1
    s = p["steps"][0]
    assert s["kind"] == "reduce" and s["reducers"] == ["sum"]
    # the whole elementwise chain is the reduction's prologue
    for op in ("multiply", "add", "tanh", "maximum", "subtract"):
        assert op in s["ops"]
    assert s["inputs"] == [0, 1]  # x and y read once; splat constants inlined
    assert p["constants"] == []


def test_c2_siblings_fuse_into_one_kernel(plugin):
    p = plan(plugin, programs.c2_argmax_f16_reductions(64, 128256))
    assert len(p["steps"]) == 1
    s = p["steps"][0]
    assert sorted(s["reducers"]) == ["argmax", "max", "min", "sum"]
    assert s["epilogue"] == ["convert"]  # f32 sum -> f16 inside the kernel
    assert s["inputs"] == [0]            # iota synthesized, not read
    assert len(s["outputs"]) == 5
    assert s["splits"] > 1 and s["grid"] >= 256  # 64 rows spread over the chip


def test_full_reduce_and_middle_axis(plugin):
    b = Builder()
    x = b.param((2, 3, 4), "f32")
    s_all = b.sum(x, [0, 1, 2])
    s_mid = b.sum(x, [1])
    m = b.max(x, [0, 2])
    p = plan(plugin, b.build([s_all, s_mid, m]))
    kinds = [st["kind"] for st in p["steps"]]
    assert kinds == ["reduce", "reduce", "reduce"]
    assert all(not st["row_schedule"] for st in p["steps"])


def test_multi_use_cheap_value_is_recomputed(plugin, monkeypatch):
    # softmax-like: exp(x - max) feeds both the sum and the divide (row
    # fusion off, so that the three passes stay separate steps).
    monkeypatch.setenv("PJRTX_ROW_FUSE_MAX", "0")
    b = Builder()
    x = b.param((8, 128), "f32")
    mx = b.max(x, [1])
    sh = b.subtract(x, b.broadcast_in_dim(mx, (8, 128), [0]))
    e = b.exp(sh)
    s = b.sum(e, [1])
    out = b.divide(e, b.broadcast_in_dim(s, (8, 128), [0]))
    p = plan(plugin, b.build([out]))
    kinds = [st["kind"] for st in p["steps"]]
    assert kinds == ["reduce", "reduce", "loop"]
    # exp is evaluated inside both the second reduction and the final loop
    assert "exponential" in p["steps"][1]["ops"] and "exponential" in p["steps"][2]["ops"]


def _softmax(b, x, via=None):
    mx = b.max(x, [1])
    if via is not None:
        mx = via(mx)
    e = b.exp(b.subtract(x, b.broadcast_in_dim(mx, x.shape, [0])))
    s = b.sum(e, [1])
    return b.divide(e, b.broadcast_in_dim(s, x.shape, [0]))


def test_softmax_is_one_row_kernel(plugin):
    b = Builder()
    x = b.param((8, 128), "f32")
    p = plan(plugin, b.build([_softmax(b, x)]))
    assert [st["kind"] for st in p["steps"]] == ["rowfused"]
    assert p["steps"][0]["phases"] == 3 and p["steps"][0]["rows"] == 8 and p["steps"][0]["row_len"] == 128
    # the row max and sum stay in registers: only the softmax output is stored
    assert len(p["steps"][0]["outputs"]) == 1


def test_row_fusion_refuses_reindexed_row_values(plugin):
    # the max is reversed before it is broadcast: row r would need row 7-r's
    # value, so the phases cannot share one workgroup per row.
    b = Builder()
    x = b.param((8, 128), "f32")
    p = plan(plugin, b.build([_softmax(b, x, via=lambda m: b.reverse(m, [0]))]))
    # max stays its own reduction; sum -> divide still fuse (the reversed max
    # is read from memory there, like any input).
    assert [st["kind"] for st in p["steps"]] == ["reduce", "rowfused"]
    assert p["steps"][0]["reducers"] == ["max"] and p["steps"][1]["phases"] == 2


def test_liveness_releases_intermediates(plugin, monkeypatch):
    monkeypatch.setenv("PJRTX_ROW_FUSE_MAX", "0")  # keep the max as a buffer between two steps
    b = Builder()
    x = b.param((4, 256), "f32")
    mx = b.max(x, [1])
    y = b.subtract(x, b.broadcast_in_dim(mx, (4, 256), [0]))
    s = b.sum(b.exp(y), [1])
    p = plan(plugin, b.build([s]))
    released = [v for st in p["steps"] for v in st["release_after"]]
    assert released, "the max intermediate must be released after its last use"


def test_reshape_of_materialized_value_is_alias(plugin):
    b = Builder()
    x = b.param((4, 6), "f32")
    s = b.sum(x, [1])
    r = b.reshape(s, (2, 2))
    p = plan(plugin, b.build([r]))
    assert [st["kind"] for st in p["steps"]] == ["reduce", "alias"]


def test_unsupported_op_fails_closed(plugin):
    text = """module @m {
  func.func public @main(%arg0: tensor<4xf32>) -> tensor<4xf32> {
    %0 = stablehlo.custom_call @foo(%arg0) : (tensor<4xf32>) -> tensor<4xf32>
    return %0 : tensor<4xf32>
  }
}"""
    with pytest.raises(PjrtError) as e:
        plugin.plan_json(text)
    assert e.value.code == 12 and "custom_call" in e.value.message


def test_parse_error_reports_line(plugin):
    text = "module @m {\n  func.func public @main(%arg0: tensor<4xf32>) -> tensor<4xf32> {\n    return %zz : tensor<4xf32>\n  }\n}"
    with pytest.raises(PjrtError) as e:
        plugin.plan_json(text)
    assert e.value.code == 3 and "line 3" in e.value.message


def test_private_function_calls_are_inlined(plugin):
    text = """module @jit_f attributes {mhlo.num_partitions = 1 : i32, mhlo.num_replicas = 1 : i32} {
  func.func public @main(%arg0: tensor<8xf32>) -> (tensor<8xf32> {jax.result_info = ""}) {
    %0 = call @relu(%arg0) : (tensor<8xf32>) -> tensor<8xf32>
    %1 = call @relu(%0) : (tensor<8xf32>) -> tensor<8xf32>
    return %1 : tensor<8xf32>
  }
  func.func private @relu(%arg0: tensor<8xf32>) -> tensor<8xf32> {
    %cst = stablehlo.constant dense<0.000000e+00> : tensor<f32>
    %0 = stablehlo.broadcast_in_dim %cst, dims = [] : (tensor<f32>) -> tensor<8xf32>
    %1 = stablehlo.maximum %arg0, %0 : tensor<8xf32>
    return %1 : tensor<8xf32>
  }
}"""
    p = plan(plugin, text)
    assert len(p["steps"]) == 1 and p["steps"][0]["kind"] == "loop"
    assert p["steps"][0]["ops"].count("maximum") == 2


def test_multi_partition_module_rejected_at_compile(plugin):
    text = programs.c1_elementwise_rowsum(4, 64).replace("mhlo.num_partitions = 1", "mhlo.num_partitions = 2")
    # planning alone accepts it; the PJRT compile path rejects (one device)
    plan(plugin, text)


@pytest.mark.parametrize("text_fn", [
    lambda: programs.c1_elementwise_rowsum(64, 256),
    lambda: programs.c2_argmax_f16_reductions(4, 1024),
    lambda: programs.c2_argmax_f16_reductions(64, 128256),
])
def test_generated_kernels_compile_for_gfx950(plugin, text_fn):
    assert plugin.compile_check(text_fn(), "gfx950") > 0


def test_generated_code_has_no_packed_f32(plugin):
    src = plugin.kernel_source(programs.c1_elementwise_rowsum(64, 256))
    assert "v_pk_" not in src
    assert "pjrtx_fusion_reduce_0" in src


def test_decode_dots_sharing_an_lhs_form_groups(plugin, monkeypatch):
    from pjrtx_amd import llama_like as L
    steps = plan(plugin, L.decode_program(L.TINY))["steps"]
    groups = [s["members"] for s in steps if s["kind"] == "gemv" and s["members"] > 1]
    assert groups == [3, 2] * L.TINY.layers  # q/k/v and gate/up of every layer
    monkeypatch.setenv("PJRTX_GEMV_FUSION", "0")
    steps = plan(plugin, L.decode_program(L.TINY))["steps"]
    groups = [s["group_size"] for s in steps if s.get("library") == "dot_group"]
    assert groups == [3, 2] * L.TINY.layers
    monkeypatch.setenv("PJRTX_DOT_GROUPS", "0")
    assert not [s for s in plan(plugin, L.decode_program(L.TINY))["steps"] if s.get("library") == "dot_group"]


def test_dot_group_refuses_a_member_that_depends_on_another(plugin):
    b = Builder()
    x = b.param((1, 64), "bf16")
    w = b.param((64, 64), "bf16")
    y = b.dot_general(x, w, contract=((1,), (0,)))
    w2 = b.multiply(w, b.broadcast_in_dim(b.reshape(y, (64,)), (64, 64), [1]))  # depends on the first dot
    z = b.dot_general(x, w2, contract=((1,), (0,)))
    steps = plan(plugin, b.build([y, z]))["steps"]
    assert "dot_group" not in [s.get("library") for s in steps]


def test_residual_add_merges_into_decode_dot(plugin, monkeypatch):
    from pjrtx_amd import llama_like as L
    steps = plan(plugin, L.decode_program(L.FULL))["steps"]
    merged = [s for s in steps if "residual_add" in s]
    assert len(merged) >= 2 * L.FULL.layers - 1  # o-proj and down-proj residuals
    assert all(s["kind"] == "gemv" for s in merged)
    monkeypatch.setenv("PJRTX_GEMV_FUSION", "0")
    steps = plan(plugin, L.decode_program(L.FULL))["steps"]
    merged = [s for s in steps if "residual_add" in s]
    assert len(merged) >= 2 * L.FULL.layers - 1
    assert all(s.get("library") == "dot_general" for s in merged)
    monkeypatch.setenv("PJRTX_DOT_RESIDUAL", "0")
    assert not [s for s in plan(plugin, L.decode_program(L.FULL))["steps"] if "residual_add" in s]


def test_decode_layer_is_five_launches(plugin):
    """Per layer: q/k/v GEMV (RMSNorm prologue, RoPE and both KV-row writes
    in its epilogue), attention, o-projection (+ residual), gate/up GEMV
    (RMSNorm prologue, SwiGLU epilogue), down projection (+ residual)."""
    from pjrtx_amd import llama_like as L
    steps = plan(plugin, L.decode_program(L.FULL))["steps"]
    units = [s for s in steps if s["kind"] != "alias"]
    gemv = [s for s in steps if s["kind"] == "gemv"]
    assert len(gemv) == 4 * L.FULL.layers + 1  # + lm_head
    qkv = [s for s in gemv if s["members"] == 3]
    assert len(qkv) == L.FULL.layers
    for s in qkv:
        assert s["prologue"] == "rowfused" and s["joint"] and s["seg_cols"] == L.FULL.head_dim
        assert "concatenate" in s["epilogue_loop"] and len(s["window_outputs"]) == 2
    up = [s for s in gemv if s["members"] == 2]
    assert all(s["prologue"] == "rowfused" and "logistic" in s["epilogue_loop"] for s in up)
    assert gemv[-1]["prologue"] == "rowfused" and gemv[-1]["N"] == [L.FULL.vocab]  # final norm + lm_head
    assert len(units) <= 5 * L.FULL.layers + 5
    # Every split GEMV folds in-launch (no combine kernel).
    assert all(s["direct"] or s["fused_combine"] for s in gemv)
    # The attention writes its 10 key splits' partials and the o-projection
    # merges them while staging its input.
    attn = [s for s in steps if s.get("library") == "attention"]
    assert len(attn) == L.FULL.layers and all(s["partials_out"] for s in attn)
    oproj = [s for s in gemv if s.get("attention_splits_merged")]
    assert len(oproj) == L.FULL.layers
    assert all(s["attention_splits_merged"] == 10 and s["members"] == 1 and "residual_add" in s for s in oproj)


def test_attention_merge_stays_in_attention_without_splits_or_when_off(plugin, monkeypatch):
    """40-slot caches give one key split: nothing to merge, the attention
    writes its rows. PJRTX_ATTN_MERGE_GEMV=0 keeps the merge in the attention
    launch."""
    from pjrtx_amd import llama_like as L
    steps = plan(plugin, L.decode_program(L.TINY))["steps"]
    assert not any(s.get("partials_out") or s.get("attention_splits_merged") for s in steps)
    monkeypatch.setenv("PJRTX_ATTN_MERGE_GEMV", "0")
    steps = plan(plugin, L.decode_program(L.FULL))["steps"]
    assert not any(s.get("partials_out") or s.get("attention_splits_merged") for s in steps)


def test_gemv_epilogue_must_stay_inside_segments(plugin):
    """A loop that reads a result across the whole row (a reverse) cannot
    run per segment: it stays its own launch."""
    b = Builder()
    x = b.param((1, 256), "bf16")
    w = b.param((256, 1024), "bf16")
    y = b.dot_general(x, w, contract=((1,), (0,)))
    z = b.multiply(b.reverse(y, [1]), y)
    steps = plan(plugin, b.build([z]))["steps"]
    assert [s["kind"] for s in steps] == ["gemv", "loop"]
    # Elementwise over the same index fuses.
    steps = plan(plugin, b.build([b.multiply(y, y)]))["steps"]
    assert [s["kind"] for s in steps] == ["gemv"] and steps[0]["epilogue_loop"] == ["multiply"]


def _shift_in_place_program():
    # c donated; c[0:7] = -c[1:8] written back into c (a roll-like shift).
    b = Builder()
    c = b.param((8, 16), "f32", donate=True)
    u = b.negate(b.slice(c, [1, 0], [8, 16]))
    z = b.constant(0, "s32")
    return b.build([b.dynamic_update_slice(c, u, [z, z])])


def test_window_write_not_absorbed_into_kernel_reading_operand(plugin):
    # The kernel computing the update reads the operand at other rows than it
    # would write: fusing the window write would race across workgroups.
    steps = plan(plugin, _shift_in_place_program())["steps"]
    assert not any(s.get("window_outputs") for s in steps)
    dus = [s for s in steps if s.get("library") == "dynamic_update_slice"]
    assert len(dus) == 1


@pytest.mark.parametrize("dt", ["s8", "u8", "s16", "u16", "s32", "u32", "s64", "u64"])
def test_popcnt_and_clz_kernels_compile_at_every_width(plugin, dt):
    """Generated popcnt / count_leading_zeros code compiles (hiprtc, no GPU)
    for every integer width (the 32-bit popcnt once emitted an extra ')')."""
    b = Builder()
    x = b.param((4, 8), dt)
    assert plugin.compile_check(b.build([b.popcnt(x), b.clz(x)])) > 0


def _wrapped_gather(vocab, dim, n, idx_dtype="s32", add_value=None):
    """table[idx] as jnp indexing lowers it (select(i < 0, i + add, i)), with
    `add` the table's row count unless given."""
    b = Builder()
    table = b.param((vocab, dim), "bf16")
    idx = b.param((n,), idx_dtype)
    add = vocab if add_value is None else add_value
    wrapped = b.select(b.compare("LT", idx, b.scalar_like(0, idx)), b.add(idx, b.scalar_like(add, idx)), idx)
    iv = b.broadcast_in_dim(wrapped, (n, 1), [0])
    return b.build([b.gather(table, iv, offset_dims=[1], collapsed_slice_dims=[0], start_index_map=[0],
                             index_vector_dim=1, slice_sizes=[1, dim])])


@pytest.mark.parametrize("idx_dtype", ["s32", "s64"])
def test_gather_index_wrap_folds_into_the_gather(plugin, monkeypatch, idx_dtype):
    # the normalization's loop kernel goes away: the gather reads the raw
    # indices through a view and applies i < 0 ? i + rows : i itself
    p = plan(plugin, _wrapped_gather(1000, 64, 16, idx_dtype))
    assert [st["kind"] for st in p["steps"]] == ["alias", "library"]
    assert p["steps"][0]["inputs"] == [1]
    monkeypatch.setenv("PJRTX_GATHER_WRAP", "0")
    p = plan(plugin, _wrapped_gather(1000, 64, 16, idx_dtype))
    kinds = [st["kind"] for st in p["steps"]]
    assert kinds == ["loop", "library"] and "select" in p["steps"][0]["ops"]


def test_gather_index_wrap_needs_the_row_count(plugin):
    # a wrap by anything but the gathered dimension's size is not JAX's
    # normalization and stays an elementwise kernel
    p = plan(plugin, _wrapped_gather(1000, 64, 16, add_value=999))
    assert [st["kind"] for st in p["steps"]] == ["loop", "library"]


def _dot_steps(plugin, make):
    b = Builder()
    return plan(plugin, b.build(make(b)))["steps"]


def test_transposed_product_swaps_its_operands(plugin):
    def make(perm, shape=(40, 24), other=(24, 56), read_twice=False):
        def f(b):
            batch = tuple(range(len(shape) - 2))
            d = b.dot_general(b.param(shape, "bf16"), b.param(other, "bf16"), batch=(batch, batch),
                              contract=((len(shape) - 1,), (len(shape) - 2,)))
            return [b.transpose(d, perm)] + ([d] if read_twice else [])
        return f
    assert len(_dot_steps(plugin, make([1, 0]))) == 1
    assert len(_dot_steps(plugin, make([0, 2, 1], (2, 40, 24), (2, 24, 56)))) == 1
    assert len(_dot_steps(plugin, make([1, 0], read_twice=True))) == 2
    assert len(_dot_steps(plugin, make([2, 1, 0], (2, 40, 24), (2, 24, 56)))) == 2  # moves the batch too
    assert len(_dot_steps(plugin, make([1, 0], (4, 24)))) == 2                      # GEMV rows stay as they are


def test_bias_row_merges_into_the_product(plugin):
    def make(bias_shape, dims, dt="bf16"):
        def f(b):
            d = b.dot_general(b.param((40, 24), "bf16"), b.param((24, 40), "bf16"), contract=((1,), (0,)), out_dtype=dt)
            return [b.add(d, b.broadcast_in_dim(b.param(bias_shape, dt), (40, 40), dims))]
        return f
    assert len(_dot_steps(plugin, make((40,), [1]))) == 1
    assert len(_dot_steps(plugin, make((40,), [0]))) == 2        # a column
    assert len(_dot_steps(plugin, make((1, 40), [0, 1]))) == 2
    assert len(_dot_steps(plugin, make((40,), [1], "f32"))) == 2


def test_sort_writes_positions_itself(plugin):
    def make(iota_dim, first=False):
        def f(b):
            ops = [b.param((8, 64), "f32"), b.iota((8, 64), iota_dim)]
            return b.sort(ops[::-1] if first else ops, 1)
        return f
    assert [s["kind"] for s in _dot_steps(plugin, make(1))] == ["library"]
    assert len(_dot_steps(plugin, make(0))) == 2               # not the position
    assert len(_dot_steps(plugin, make(1, first=True))) == 2   # the key itself


def _top_k_step(plugin, rows, n, k, dt="bf16"):
    b = Builder()
    (step,) = plan(plugin, b.build(list(b.top_k(b.param((rows, n), dt), k))))["steps"]
    return step


def _kept_words(rows, n, k):
    """Bytes of two lists that hold the first k (rounded up to a power of two)
    of every 4096 words of 8 bytes: what a top_k over long rows may take."""
    return 2 * rows * -(-n // 4096) * (1 << (k - 1).bit_length()) * 8


@pytest.mark.parametrize("dt", ["s8", "bf16"])
@pytest.mark.parametrize("k", [1, 50, 256, 257, 2048])
def test_top_k_of_rows_that_words_cannot_number(plugin, k, dt):
    """A word holds 30 bits of position; longer rows are taken in pieces, not
    sorted whole (16 GB of words and hundreds of passes at 2^30 elements)."""
    for n in (2 ** 30 - 8, 2 ** 30, 2 ** 30 + 24, 2 ** 31 - 8):
        assert _top_k_step(plugin, 2, n, k, dt)["scratch_bytes"] <= _kept_words(2, n, k)


@pytest.mark.parametrize("rows,n,k", [(1, 8193, 256), (3, 40000, 256), (16, 32000, 64), (64, 128256, 128), (200, 20000, 1),
                                      (1, 10 ** 7, 256), (64, 128256, 300), (2, 50000, 4096), (1, 2 ** 30, 256)])
def test_top_k_takes_no_more_room_than_kept_words(plugin, rows, n, k):
    """Where scratch is a fixed block, a top_k makes do with the kept words of
    each 4096, however few workgroups that leaves."""
    assert _top_k_step(plugin, rows, n, k)["least_scratch_bytes"] <= _kept_words(rows, n, k)


def attention_then_transpose(shape, perm, dt="bf16", twice=False):
    """c3_attention whose result is transposed (and also returned, `twice`)."""
    mlir = lambda d: "tensor<" + "x".join(map(str, d)) + f"x{dt}>"  # noqa: E731
    src, dst = mlir(shape), mlir([shape[p] for p in perm])
    text = programs.c3_attention(*shape, True, dtype=dt)
    head = next(ln for ln in text.splitlines() if "func.func" in ln)
    ret = next(ln for ln in text.splitlines() if ln.strip().split(" ")[0] in ("return", "func.return", "stablehlo.return"))
    name = ret.split()[1]
    both = (f"%tr, {name} : {dst}, {src}", f"({dst}, {src})") if twice else (f"%tr : {dst}", dst)
    text = text.replace(ret, f"    %tr = stablehlo.transpose {name}, dims = {list(perm)} : ({src}) -> {dst}\n    return {both[0]}")
    return text.replace(head, head[:head.index("->")] + f"-> {both[1]} {{")


def test_attention_writes_its_transposed_result(plugin):
    kinds = lambda *a, **k: [s.get("library", s["kind"]) for s in plan(plugin, attention_then_transpose(*a, **k))["steps"]]  # noqa: E731
    assert kinds((2, 4, 128, 64), [0, 2, 1, 3]) == ["attention"]
    assert kinds((2, 4, 128, 64), [0, 2, 1, 3], twice=True) == ["attention", "loop"]
    assert kinds((2, 4, 128, 64), [0, 1, 3, 2]) == ["attention", "loop"]
    assert kinds((2, 4, 8, 64), [0, 2, 1, 3]) == ["attention", "loop"]  # few queries


@pytest.mark.parametrize("lhs,rhs,contract,add,stride", [
    ((64, 128), (128, 8, 32), ((1,), (0,)), None, 256),            # heads and head dim: both are columns
    ((512, 128), (512, 8, 32), ((0,), (0,)), None, 256),           # a [d, heads, head_dim] weight's gradient
    ((4096, 128), (128,), ((1,), (0,)), None, 1),                  # a vector: one column
    ((64, 128), (128, 2, 3, 4), ((1,), (0,)), None, 24),
    ((16, 4, 128), (128, 40), ((2,), (0,)), None, 40),             # rows of two dims
    ((64, 128), (8, 128, 32), ((1,), (1,)), None, 256),            # columns that are apart
    ((64, 128), (128, 40), ((1,), (0,)), "row", 0),
])
def test_merged_addend_rows_are_the_products(plugin, lhs, rhs, contract, add, stride):
    """An addend of the result's shape is read a product row at a time: its row
    stride is all of the right operand's free dims, not the last one."""
    b = Builder()
    d = b.dot_general(b.param(lhs, "bf16"), b.param(rhs, "bf16"), contract=contract)
    x = b.broadcast_in_dim(b.param((rhs[-1],), "bf16"), d.shape, [len(d.shape) - 1]) if add else b.param(d.shape, "bf16")
    (step,) = plan(plugin, b.build([b.add(d, x)]))["steps"]
    assert step["residual_stride"] == stride


@pytest.mark.parametrize("rhs,batch,stride", [((3, 128), ((0,), (0,)), 1), ((3, 128, 4, 8), ((0,), (0,)), 32)])
def test_merged_addend_rows_of_batched_products(plugin, rhs, batch, stride):
    b = Builder()
    d = b.dot_general(b.param((3, 40, 128), "bf16"), b.param(rhs, "bf16"), batch=batch, contract=((2,), (1,)))
    (step,) = plan(plugin, b.build([b.add(b.param(d.shape, "bf16"), d)]))["steps"]
    assert step["residual_stride"] == stride


@pytest.mark.parametrize("dims", [[0], [1]])
def test_vector_accesses_take_64_bit_positions(plugin, dims):
    """Past 2^32 elements a position does not fit 32 bits: the vector loads
    and stores take the kernel's index type as it is."""
    b = Builder()
    x = b.param((65537, 65536), "bf16")
    src = plugin.kernel_source(b.build([b.max(x, dims), b.add(x, x)]))
    assert "typedef uint64_t idx_t" in src and "typedef uint32_t idx_t" not in src and "ldv<" in src and "stv<" in src
    for fn in ("ldv", "stv"):
        (sig,) = re.findall(r"PJRTX_DEV void %s\((.*)\) \{" % fn, src)
        assert "uint32_t base" not in sig and "I base" in sig


def _operands(plugin, lhs, rhs, contract, batch=((), ())):
    b = Builder()
    d = b.dot_general(b.param(lhs, "bf16"), b.param(rhs, "bf16"), batch=batch, contract=contract)
    (step,) = plan(plugin, b.build([d]))["steps"]
    return step["operands"]


@pytest.mark.parametrize("lhs,rhs,contract,scalar", [
    ((256, 9), (9, 256), ((1,), (0,)), True),            # padded first, 2.6 us more a launch
    ((256, 9), (256, 9), ((1,), (1,)), True),
    ((256, 28), (256, 28), ((1,), (1,)), True),          # both padded
    ((256, 28), (28, 256), ((1,), (0,)), False),         # one
    ((256, 44), (256, 44), ((1,), (1,)), False),
    ((256, 8), (8, 256), ((1,), (0,)), False),           # nothing to pad
    ((12, 256), (12, 256), ((0,), (0,)), False),
    ((5, 256), (5, 256), ((0,), (0,)), True),            # less than a k-tile's launch
    ((512, 2), (4096, 2), ((1,), (1,)), True),
    ((1000, 5), (5, 520), ((1,), (0,)), True),
    ((4096, 5), (5, 4096), ((1,), (0,)), False),         # too many results
    ((3, 9), (9, 8192), ((1,), (0,)), True),             # decode rows: the GEMV of a ragged K
    ((1, 9), (9, 8192), ((1,), (0,)), False),
    ((3, 64), (64, 8192), ((1,), (0,)), False),
])
def test_small_ragged_products_go_to_the_scalar_kernel(plugin, lhs, rhs, contract, scalar):
    b = Builder()
    d = b.dot_general(b.param(lhs, "bf16"), b.param(rhs, "bf16"), contract=contract)
    (step,) = plan(plugin, b.build([d]))["steps"]
    assert step.get("scalar", False) is scalar


def test_operands_are_read_within_their_bounds(plugin):
    """The block tiles read whole 16-byte pieces: an operand whose only row
    ends inside one (an outer product's right side) is padded like ragged rows."""
    assert _operands(plugin, (64, 40), (40, 24), ((1,), (0,))) == ["read", "read"]
    assert _operands(plugin, (64, 40), (40, 23), ((1,), (0,))) == ["read", "padded"]
    assert _operands(plugin, (40, 64), (40, 24), ((0,), (0,))) == ["read", "read"]
    assert _operands(plugin, (64, 1), (1, 24), ((1,), (0,))) == ["padded", "read"]
    assert _operands(plugin, (64, 1), (1, 23), ((1,), (0,))) == ["padded", "padded"]
    assert _operands(plugin, (64,), (23,), ((), ())) == ["padded", "padded"]
    assert _operands(plugin, (3, 64, 1), (3, 1, 24), ((2,), (1,)), ((0,), (0,))) == ["padded", "read"]


@pytest.mark.parametrize("lhs,rhs,contract,tiles", [
    ((1 << 20, 64), (64, 1 << 15), ((1,), (0,)), True),        # a 64 GB result: 2^24 of the smallest tiles
    ((64, 1 << 22), ((1 << 22), 64), ((1,), (0,)), False),     # rows of 4M elements
    ((64, (1 << 22) - 8), ((1 << 22) - 8, 64), ((1,), (0,)), True),
    ((1 << 22, 64), (1 << 22, 64), ((0,), (0,)), True),        # contracted over long columns
])
def test_sizes_of_the_block_tiles(plugin, lhs, rhs, contract, tiles):
    b = Builder()
    d = b.dot_general(b.param(lhs, "bf16"), b.param(rhs, "bf16"), contract=contract)
    (step,) = plan(plugin, b.build([d]))["steps"]
    assert step["block_tiles"] is tiles


def test_few_ragged_columns_are_transposed_for_decode_rows(plugin):
    """The K-contiguous GEMV is the faster one there (2048 x 257: 8.8 us, 12.7
    padded for the tiles)."""
    kn = ((1,), (0,))
    assert _operands(plugin, (1, 2048), (2048, 257), kn) == ["read", "copied"]
    assert _operands(plugin, (4, 512), (512, 10), kn) == ["read", "copied"]
    assert _operands(plugin, (5, 2048), (2048, 257), kn) == ["read", "padded"]
    assert _operands(plugin, (1, 2048), (2048, 513), kn) == ["read", "padded"]
    assert _operands(plugin, (1, 2044), (2044, 257), kn) == ["padded", "padded"]
    assert _operands(plugin, (1, 2048), (257, 2048), ((1,), (1,))) == ["read", "read"]


def test_dims_of_one_element_do_not_merge_their_neighbours(plugin):
    """Free (or contracted) dims are one stride only where the dims of more
    than one element follow each other; one of 1 between them changes nothing."""
    assert _operands(plugin, (2, 40, 1, 8), (40, 24), ((1,), (0,))) == ["copied", "read"]
    assert _operands(plugin, (2, 40, 8), (40, 24), ((1,), (0,))) == ["copied", "read"]
    assert _operands(plugin, (2, 1, 8, 40), (40, 24), ((3,), (0,))) == ["read", "read"]
    assert _operands(plugin, (64, 2, 20), (2, 24, 1, 20), ((1, 2), (0, 3))) == ["read", "copied"]
    assert _operands(plugin, (64, 1, 2, 20), (1, 2, 20, 24), ((1, 2, 3), (0, 1, 2))) == ["read", "read"]


@pytest.mark.parametrize("shape,inputs,lanes", [
    ((1024, 4096), ["f32"], "64"), ((256, 65536), ["f32"], "64"), ((64, 1 << 22), ["f32"], "64"),
    ((64, 1 << 20), ["bf16"], 0),              # what the memory-side cache holds
    ((1024, 65540), ["f32"], 0), ((1024, 65537), ["bf16"], 0), ((32, 65537), ["f32"], "64"),
    ((256, 65536), ["bf16", "f32", "f32"], 0), ((256, 40960), ["bf16", "f32", "f32"], "64"),
    ((1024, 40001), ["f32"], 256), ((1024, 9001), ["f32"], "64"), ((100, 40001), ["f32"], "64"),
    ((64, 1), ["f32"], 8), ((200, 16), ["bf16"], 8),  # short columns of few outputs: 32 lane rows
])
def test_schedule_of_column_reductions(plugin, shape, inputs, lanes):
    """Lanes that span outputs, or one serial thread an output where that
    streams whole rows better."""
    b = Builder()
    x = [b.param(shape, dt) for dt in inputs]
    total = b.convert(x[0], "f32") if inputs[0] != "f32" else x[0]
    for y in x[1:]:
        total = b.add(total, y)
    (step,) = plan(plugin, b.build([b.sum(total, [0])]))["steps"]
    assert not step["row_schedule"]
    assert 8 <= step["column_lanes"] <= 64 if lanes == "64" else step["column_lanes"] == lanes
