"""The work that programs hand to the plugin, as cases that can be timed and
checked: StableHLO programs compiled through the PJRT client and executed on
buffers that are already on the GPU.

A case is a dict with a "kind" and its sizes. The kinds, and what each stands
for in real use:

  rowsum     an elementwise chain with a row reduction, f32 (a fused loss or
             norm term)
  argmax     greedy decoding's choice over the logits with the f16 sum, max
             and min of the same row
  matmul     a plain product, from a few rows to square
  linear     a dense layer in training: forward, and the gradients of its
             input, weight and bias, as jax.vjp of x @ w + b lowers them
  attention  softmax attention over whole sequences (prefill)
  gather     an embedding lookup
  scatter    an embedding's gradient or a histogram: rows added at indices
             with heavy duplicates, in update order
  prefill    a llama-like decoder over a prompt: logits and caches
  decode     one token of the same decoder at batch 1: logits and caches
  topk       the candidate set of top-k sampling over logits
  argsort    a stable sort of rows with their positions (top-p sampling,
             ranking)

`prepare` uploads the inputs, as a program does before its loop, and compiles
the program; `run` is one PJRT execute. Its results are handed back as torch
views of the result buffers (no copy).
"""
import ctypes
import math

import numpy as np
import torch

from pjrtx_amd import llama_like, programs
from pjrtx_amd.hlo import Builder
from pjrtx_amd.pjrt import Client

_TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "s32": torch.int32}
_SIZE = {"bf16": 2, "f16": 2, "f32": 4, "s32": 4}


# ------------------------------------------------------------------- cases

def listed():
    return [
        # The elementwise and reduction benchmark, at its full size.
        {"name": "rowsum_4096x4096", "kind": "rowsum", "rows": 4096, "cols": 4096},
        # The smallest call: one launch of a few microseconds, so launch and
        # client costs count.
        {"name": "argmax_64x128256", "kind": "argmax", "rows": 64, "cols": 128256},
        # The largest product of the benchmark.
        {"name": "matmul_8192", "kind": "matmul", "m": 8192, "k": 8192, "n": 8192, "dtype": "bf16"},
        # A training step's dense layer; the token count is no multiple of a tile.
        {"name": "linear_1000x2048x5632", "kind": "linear", "tokens": 1000, "d_in": 2048, "d_out": 5632},
        # The attention benchmark.
        {"name": "attention_8x32x2048x128", "kind": "attention", "batch": 8, "heads": 32, "seq": 2048,
         "head_dim": 128, "causal": True},
        # The embedding lookup of a large vocabulary.
        {"name": "gather_16384_of_128256", "kind": "gather", "vocab": 128256, "dim": 4096, "batch": 8, "seq": 2048},
        # The scatter-add benchmark in both its types.
        {"name": "scatter_f32_1048576", "kind": "scatter", "rows": 65536, "dim": 256, "updates": 1048576,
         "dtype": "f32"},
        {"name": "scatter_s32_1048576", "kind": "scatter", "rows": 65536, "dim": 256, "updates": 1048576,
         "dtype": "s32"},
        # The decoder's two whole calls, in the benchmark's configuration.
        {"name": "prefill_512", "kind": "prefill", "layers": 8, "d_model": 2048, "ffn": 5632, "vocab": 32000,
         "prompt": 512, "max_len": 640},
        {"name": "decode_at_600", "kind": "decode", "layers": 8, "d_model": 2048, "ffn": 5632, "vocab": 32000,
         "pos": 600, "max_len": 640},
        # Sampling.
        {"name": "topk_50_of_128256", "kind": "topk", "rows": 64, "cols": 128256, "k": 50},
        {"name": "argsort_64x32000", "kind": "argsort", "rows": 64, "cols": 32000, "dtype": "f32"},
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm; half of them of the
    round sizes that models have, the others any."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 64 and rng.random() < 0.5:
        unit = 64 if v < 4096 else 256
        v = v // unit * unit
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["rowsum", "argmax", "matmul", "linear", "attention", "gather", "scatter", "prefill", "decode",
                       "topk", "argsort"])
    while True:
        c = _draw(kind, rng)
        if c is not None:
            return c


def _draw(kind, rng):
    """A case of the kind, or None where it would cost more than the listed ones."""
    if kind == "rowsum":
        c = {"kind": kind, "rows": _log_int(rng, 16, 16384), "cols": _log_int(rng, 256, 16384)}
        return c if c["rows"] * c["cols"] <= 4096 * 4096 else None
    if kind == "argmax":
        c = {"kind": kind, "rows": _log_int(rng, 1, 512), "cols": _log_int(rng, 4000, 160000)}
        return c if c["rows"] * c["cols"] <= 1 << 26 else None
    if kind == "matmul":
        c = {"kind": kind, "m": _log_int(rng, 1, 8192), "k": _log_int(rng, 256, 8192), "n": _log_int(rng, 256, 8192),
             "dtype": rng.choice(["bf16", "bf16", "bf16", "f16"])}
        return c
    if kind == "linear":
        c = {"kind": kind, "tokens": _log_int(rng, 64, 8192), "d_in": _log_int(rng, 512, 8192),
             "d_out": _log_int(rng, 512, 8192)}
        return c if c["tokens"] * c["d_in"] * c["d_out"] <= 1 << 37 else None
    if kind == "attention":
        c = {"kind": kind, "batch": rng.randint(1, 8), "heads": rng.choice([4, 8, 12, 16, 32]),
             "seq": _log_int(rng, 32, 2048), "head_dim": rng.choice([64, 128]), "causal": rng.random() < 0.7}
        return c
    if kind == "gather":
        c = {"kind": kind, "vocab": _log_int(rng, 1000, 128256), "dim": _log_int(rng, 64, 4096),
             "batch": rng.randint(1, 8), "seq": _log_int(rng, 1, 2048)}
        return c
    if kind == "scatter":
        c = {"kind": kind, "rows": _log_int(rng, 256, 65536), "dim": _log_int(rng, 16, 1024),
             "updates": _log_int(rng, 1024, 1048576), "dtype": rng.choice(["f32", "s32"])}
        return c if c["updates"] * c["dim"] <= 1 << 27 else None
    if kind in ("prefill", "decode"):
        d = rng.choice([512, 1024, 2048])
        c = {"kind": kind, "layers": rng.randint(1, 8), "d_model": d, "ffn": rng.choice([2 * d, 11 * d // 4, 4 * d]),
             "vocab": _log_int(rng, 2000, 32000)}
        if c["layers"] * c["ffn"] > 8 * 5632:
            return None
        if kind == "prefill":
            c["prompt"] = _log_int(rng, 16, 512)
            c["max_len"] = c["prompt"] + rng.randint(1, 128)
        else:
            c["max_len"] = _log_int(rng, 64, 2048)
            c["pos"] = rng.randint(0, c["max_len"] - 1)
        return c
    if kind == "topk":
        c = {"kind": kind, "rows": _log_int(rng, 1, 256), "cols": _log_int(rng, 2000, 160000),
             "k": rng.choice([1, 5, 10, 20, 40, 50, 64, 100, 200])}
        return c if c["rows"] * c["cols"] <= 64 * 128256 else None
    c = {"kind": kind, "rows": _log_int(rng, 1, 4096), "cols": _log_int(rng, 100, 200000),
         "dtype": rng.choice(["f32", "f32", "bf16", "s32"])}
    return c if c["rows"] * c["cols"] <= 64 * 32000 else None


# ---------------------------------------------------------------- programs

def _linear_program(t, d_in, d_out):
    """jax.vjp of x @ w + b (b broadcast over the tokens), jitted: the weight
    gradient is dot_general(g, x) transposed, the bias gradient a bf16 sum
    over the tokens (accumulated in f32)."""
    b = Builder("jit_linear")
    x, w = b.param((t, d_in), "bf16"), b.param((d_in, d_out), "bf16")
    bias, g = b.param((d_out,), "bf16"), b.param((t, d_out), "bf16")
    y = b.dot_general(x, w, contract=((1,), (0,)))
    y = b.add(y, b.broadcast_in_dim(bias, y.shape, [1]))
    dx = b.dot_general(g, w, contract=((1,), (1,)))
    dw = b.transpose(b.dot_general(g, x, contract=((0,), (0,))), [1, 0])
    db = b.sum(g, [0])
    return b.build([y, dx, dw, db])


def _argsort_program(rows, cols, dtype):
    b = Builder("jit_argsort")
    x = b.param((rows, cols), dtype)
    v, i = b.sort([x, b.iota((rows, cols), 1)], 1)
    return b.build([v, i])


def _llama(c):
    return llama_like.LlamaConfig(layers=c["layers"], d_model=c["d_model"], heads=c["d_model"] // 128, head_dim=128,
                                  ffn=c["ffn"], vocab=c["vocab"], max_len=c["max_len"],
                                  prompt=c.get("prompt", 1))


def _program(c):
    kind = c["kind"]
    if kind == "rowsum":
        return programs.c1_elementwise_rowsum(c["rows"], c["cols"])
    if kind == "argmax":
        return programs.c2_argmax_f16_reductions(c["rows"], c["cols"])
    if kind == "matmul":
        return programs.c3_matmul(c["m"], c["k"], c["n"], c["dtype"])
    if kind == "linear":
        return _linear_program(c["tokens"], c["d_in"], c["d_out"])
    if kind == "attention":
        return programs.c3_attention(c["batch"], c["heads"], c["seq"], c["head_dim"], c["causal"])
    if kind == "gather":
        return programs.c4_embedding_gather(c["vocab"], c["dim"], c["batch"], c["seq"])
    if kind == "scatter":
        return programs.c4_scatter_add(c["rows"], c["dim"], c["updates"], c["dtype"])
    if kind == "prefill":
        return llama_like.prefill_program(_llama(c))
    if kind == "decode":
        return llama_like.decode_program(_llama(c))
    if kind == "topk":
        return programs.topk_logits(c["rows"], c["cols"], c["k"])
    return _argsort_program(c["rows"], c["cols"], c["dtype"])


# ------------------------------------------------------------------ inputs

def _inputs(c, seed):
    """The arguments as torch tensors on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(shape, dtype, scale=1.0):
        return torch.randn(shape, device="cuda", generator=g).mul_(scale).to(_TORCH[dtype])

    kind = c["kind"]
    if kind == "rowsum":
        shape = (c["rows"], c["cols"])
        return [torch.rand(shape, device="cuda", generator=g).mul_(2).sub_(1) for _ in range(2)]
    if kind == "argmax":
        return [normal((c["rows"], c["cols"]), "bf16")]
    if kind == "matmul":
        s = c["k"] ** -0.25
        return [normal((c["m"], c["k"]), c["dtype"], s), normal((c["k"], c["n"]), c["dtype"], s)]
    if kind == "linear":
        t, i, o = c["tokens"], c["d_in"], c["d_out"]
        return [normal((t, i), "bf16"), normal((i, o), "bf16", i ** -0.5), normal((o,), "bf16", 0.02),
                normal((t, o), "bf16", 0.1)]
    if kind == "attention":
        shape = (c["batch"], c["heads"], c["seq"], c["head_dim"])
        return [normal(shape, "bf16", c["head_dim"] ** -0.5) for _ in range(3)]
    if kind == "gather":
        return [normal((c["vocab"], c["dim"]), "bf16", 0.02),
                torch.randint(0, c["vocab"], (c["batch"], c["seq"]), device="cuda", generator=g, dtype=torch.int32)]
    if kind == "scatter":
        idx = ((np.random.default_rng(seed).zipf(1.1, c["updates"]) - 1) % c["rows"]).astype(np.int32)
        shape = (c["updates"], c["dim"])
        if c["dtype"] == "f32":
            upd = normal(shape, "f32")
        else:
            upd = torch.randint(-1000, 1000, shape, device="cuda", generator=g, dtype=torch.int32)
        return [torch.zeros((c["rows"], c["dim"]), device="cuda", dtype=upd.dtype), torch.from_numpy(idx).cuda(), upd]
    if kind in ("prefill", "decode"):
        cfg = _llama(c)
        args = []
        for name, shape in llama_like.weight_shapes(cfg):
            args.append(torch.ones(shape, device="cuda", dtype=torch.bfloat16) if name.endswith("norm")
                        else normal(shape, "bf16", 0.02))
        cache = llama_like.cache_shape(cfg)
        if kind == "prefill":
            args.append(torch.randint(0, cfg.vocab, (cfg.prompt,), device="cuda", generator=g, dtype=torch.int32))
            return args + [torch.zeros(cache, device="cuda", dtype=torch.bfloat16) for _ in range(2 * cfg.layers)]
        args.append(torch.randint(0, cfg.vocab, (1,), device="cuda", generator=g, dtype=torch.int32))
        args.append(torch.tensor(c["pos"], dtype=torch.int32, device="cuda"))
        for _ in range(2 * cfg.layers):  # keys and values of the positions before this one
            t = normal(cache, "bf16", 0.9)
            t[:, :, c["pos"]:] = 0
            args.append(t)
        return args
    if kind == "topk":
        return [normal((c["rows"], c["cols"]), "bf16", 2.0)]
    if c["dtype"] == "s32":
        return [torch.randint(-(1 << 31), (1 << 31) - 1, (c["rows"], c["cols"]), device="cuda", generator=g,
                              dtype=torch.int32)]
    return [normal((c["rows"], c["cols"]), c["dtype"], 2.0)]


_client = None


def client():
    """The process's PJRT client."""
    global _client
    if _client is None:
        _client = Client()
    return _client


def _upload(t):
    if t.dtype == torch.bfloat16:
        return client().buffer(t.view(torch.int16).cpu().numpy().view(np.uint16), "bf16")
    return client().buffer(t.cpu().numpy())


class _PointerArgs(ctypes.Structure):
    """PJRT_Buffer_OpaqueDeviceMemoryDataPointer_Args (include/pjrt_c_api.h)."""
    _fields_ = [("struct_size", ctypes.c_size_t), ("extension_start", ctypes.c_void_p), ("buffer", ctypes.c_void_p),
                ("device_memory_ptr", ctypes.c_void_p)]


class _View:
    """A result buffer for torch.as_tensor, which keeps this object (and with
    it the buffer) as long as the tensor lives."""

    def __init__(self, buf, shape, typestr):
        a = _PointerArgs(struct_size=ctypes.sizeof(_PointerArgs), buffer=buf.handle)
        buf.client.p.call("Buffer_OpaqueDeviceMemoryDataPointer", a)
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (a.device_memory_ptr, False),
                                         "strides": None, "version": 2}


_TYPESTR = {"bf16": "<i2", "f16": "<f2", "f32": "<f4", "s32": "<i4"}


def _tensor(buf, spec):
    shape, dtype = spec
    t = torch.as_tensor(_View(buf, shape, _TYPESTR[dtype]), device="cuda")
    return t.view(torch.bfloat16) if dtype == "bf16" else t


def _result_specs(c):
    """Shape and type of each result that `run` hands back."""
    kind = c["kind"]
    if kind == "rowsum":
        return [((c["rows"],), "f32")]
    if kind == "argmax":
        r = (c["rows"],)
        return [(r, "bf16"), (r, "s32"), (r, "f16"), (r, "f16"), (r, "f16")]
    if kind == "matmul":
        return [((c["m"], c["n"]), c["dtype"])]
    if kind == "linear":
        t, i, o = c["tokens"], c["d_in"], c["d_out"]
        return [((t, o), "bf16"), ((t, i), "bf16"), ((i, o), "bf16"), ((o,), "bf16")]
    if kind == "attention":
        return [((c["batch"], c["heads"], c["seq"], c["head_dim"]), "bf16")]
    if kind == "gather":
        return [((c["batch"], c["seq"], c["dim"]), "bf16")]
    if kind == "scatter":
        return [((c["rows"], c["dim"]), c["dtype"])]
    if kind in ("prefill", "decode"):
        cfg = _llama(c)
        return [((1, cfg.vocab), "bf16")] + [(llama_like.cache_shape(cfg), "bf16")] * (2 * cfg.layers)
    if kind == "topk":
        return [((c["rows"], c["k"]), "bf16"), ((c["rows"], c["k"]), "s32")]
    return [((c["rows"], c["cols"]), c["dtype"]), ((c["rows"], c["cols"]), "s32")]


def prepare(case, seed):
    args = [_upload(t) for t in _inputs(case, seed)]
    state = {"exe": client().compile(_program(case)), "args": args, "caches": [], "skip": 0,
             "specs": _result_specs(case)}
    if case["kind"] in ("prefill", "decode"):
        # The caches are donated: each call hands its own back. The first
        # result is the next token, the arg-max of the logits: with random
        # weights the best two are often a rounding apart, so the logits are
        # what is compared.
        n = 2 * case["layers"]
        state.update(args=args[:-n], caches=args[-n:], skip=1)
    return state


def run(state):
    outs = state["exe"].execute_buffers(state["args"] + state["caches"])
    outs = outs[state["skip"]:]
    if state["caches"]:
        state["caches"] = outs[1:]
    return [_tensor(b, s) for b, s in zip(outs, state["specs"])]


# ------------------------------------------------------- work and tolerance

def work(case):
    c, kind = case, case["kind"]
    if kind == "rowsum":
        n = c["rows"] * c["cols"]
        return {"bytes": 8 * n + 4 * c["rows"], "flops": 7 * n}
    if kind == "argmax":
        n = c["rows"] * c["cols"]
        return {"bytes": 2 * n + 12 * c["rows"], "flops": 4 * n}
    if kind == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": 2 * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "linear":
        t, i, o = c["tokens"], c["d_in"], c["d_out"]
        return {"bytes": 2 * (2 * t * i + 2 * i * o + 2 * t * o + 2 * o), "flops": 6 * t * i * o}
    if kind == "attention":
        s = c["seq"]
        pairs = s * (s + 1) // 2 if c["causal"] else s * s
        bh = c["batch"] * c["heads"]
        return {"bytes": 8 * bh * s * c["head_dim"], "flops": 4 * bh * pairs * c["head_dim"]}
    if kind == "gather":
        n = c["batch"] * c["seq"]
        return {"bytes": n * (4 + 4 * c["dim"]), "flops": 0}
    if kind == "scatter":
        return {"bytes": 4 * c["updates"] * (c["dim"] + 1) + 8 * c["rows"] * c["dim"],
                "flops": c["updates"] * c["dim"]}
    if kind in ("prefill", "decode"):
        cfg = _llama(c)
        n = cfg.prompt if kind == "prefill" else 1
        d, q, f = cfg.d_model, cfg.qdim, cfg.ffn
        layer = 4 * d * q + 3 * d * f
        weights = cfg.layers * (layer + 2 * d) + d + d * cfg.vocab + n * d
        keys = n * (n + 1) // 2 if kind == "prefill" else c["pos"] + 1
        rows = 2 * n if kind == "prefill" else 2 * (c["pos"] + 2)  # cache rows written, and at decode read
        return {"bytes": 2 * (weights + cfg.layers * rows * q + cfg.vocab),
                "flops": 2 * (n * cfg.layers * layer + d * cfg.vocab) + 4 * cfg.layers * keys * q}
    if kind == "topk":
        return {"bytes": c["rows"] * (2 * c["cols"] + 6 * c["k"]), "flops": 0}
    return {"bytes": c["rows"] * c["cols"] * (2 * _SIZE[c["dtype"]] + 4), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "rowsum":
        return {"rel": 1e-5, "max": 1e-4}        # f32 sums in another order
    if kind == "argmax":
        return {"rel": 1e-3, "max": 4e-3}        # the f16 sum's rounding; the rest is exact
    if kind in ("matmul", "linear"):
        return {"rel": 5e-3, "max": 4e-2}        # one bf16 rounding of an f32 sum
    if kind == "attention":
        return {"rel": 1e-2, "max": 0.1}         # bf16 probabilities, one bf16 rounding of the result
    if kind in ("prefill", "decode"):
        return {"rel": 3e-2, "max": 0.5}         # bf16 roundings carried through the layers (2% off 64 bits)
    return "exact"                               # selections, and sums in update order


# -------------------------------------------------------------------- exact

def _exact_llama(c, args):
    """The decoder in 64 bits, with no rounding between its operations."""
    cfg = _llama(c)
    names = [n for n, _ in llama_like.weight_shapes(cfg)]
    w = dict(zip(names, args))
    n = cfg.prompt if c["kind"] == "prefill" else 1
    start = 0 if c["kind"] == "prefill" else c["pos"]
    rest = args[len(names) + (1 if c["kind"] == "prefill" else 2):]
    caches = [t.double() for t in rest]
    tokens = args[len(names)].long()
    pos = torch.arange(start, start + n, device="cuda")
    inv = torch.from_numpy(llama_like.rope_inv_freq(cfg)).cuda().double()
    ang = pos.double()[:, None] * inv[None]
    cos, sin = torch.cat([ang.cos()] * 2, 1), torch.cat([ang.sin()] * 2, 1)

    def norm(x, gain):
        return x * torch.rsqrt((x * x).sum(1, keepdim=True) / cfg.d_model + cfg.eps) * gain.double()

    def heads(x):
        return x.view(n, cfg.heads, cfg.head_dim).transpose(0, 1).contiguous()

    def rope(x):
        half = cfg.head_dim // 2
        return x * cos + torch.cat([-x[..., half:], x[..., :half]], 2) * sin

    x = w["embed"][tokens].double()
    for i in range(cfg.layers):
        g = lambda name: w["l%d.%s" % (i, name)].double()  # noqa: E731
        h = norm(x, g("attn_norm"))
        q, k, v = rope(heads(h @ g("wq"))), rope(heads(h @ g("wk"))), heads(h @ g("wv"))
        kc, vc = caches[2 * i][0], caches[2 * i + 1][0]
        kc[:, start:start + n], vc[:, start:start + n] = k, v
        s = torch.matmul(q, kc.transpose(1, 2).contiguous()) / math.sqrt(cfg.head_dim)
        s.masked_fill_(torch.arange(cfg.max_len, device="cuda")[None, :] > pos[:, None], -math.inf)
        ctx = torch.matmul(torch.softmax(s, 2), vc)
        x = x + ctx.transpose(0, 1).reshape(n, cfg.qdim) @ g("wo")
        h = norm(x, g("ffn_norm"))
        a = h @ g("w1")
        x = x + (a * torch.sigmoid(a) * (h @ g("w3"))) @ g("w2")
    return [norm(x[-1:], w["final_norm"]) @ w["lm_head"].double()] + caches


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("gather", "topk", "argsort"):
        return None  # values of the input, in another place
    args = _inputs(c, seed)
    if kind == "rowsum":
        x, y = (t.double() for t in args)
        return [(torch.tanh(x * y + 0.5) * x - y.clamp(min=0)).sum(1)]
    if kind == "argmax":
        x = args[0]
        h = x.to(torch.float16).double()
        return [x.double().amax(1), None, h.sum(1), h.amax(1), h.amin(1)]
    if kind == "matmul":
        return [args[0].double() @ args[1].double()]
    if kind == "linear":
        x, w, b, g = (t.double() for t in args)
        return [x @ w + b, g @ w.t(), x.t() @ g, g.sum(0)]
    if kind == "attention":
        q, k, v = args
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        mask = torch.ones(c["seq"], c["seq"], dtype=torch.bool, device="cuda").triu(1)
        for i in range(c["batch"]):
            for h in range(c["heads"]):
                s = q[i, h].double() @ k[i, h].double().t()
                if c["causal"]:
                    s.masked_fill_(mask, -math.inf)
                out[i, h] = torch.softmax(s, 1) @ v[i, h].double()
        return [out]
    if kind == "scatter":
        x, idx, upd = args
        if c["dtype"] == "s32":
            return None  # whole numbers
        out = x.double()
        step = max(1, (1 << 27) // c["dim"])
        for lo in range(0, c["updates"], step):
            out.index_add_(0, idx[lo:lo + step].long(), upd[lo:lo + step].double())
        return [out]
    return _exact_llama(c, args)
