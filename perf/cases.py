"""The work a program has this framework do, as cases that can be timed and compared.

Five kinds of case, each through the entry points a program calls (the C-ABI's recordings
and replays by way of skyla_hip.engine):

  matvecs   the decode matrix-vector products of a stack of layers (Graph.matvec, one token):
            q, k, v, o, gate, up, down of each layer, every layer its own weights
  matmuls   the same products of one layer over the token rows of a prefill chunk or batch
  moe       a mixture-of-experts layer (Graph.moe): decode (one token) and prefill chunks
  step      Engine.step: one token through a model, at a position of a filled KV cache
  prefill   Engine.prefill: a prompt, after a position of the cache

Sizes are those of the benchmark's and tests' models (Qwen3-0.6B in Q8_0, Qwen3-8B in
Q4_K with Q6_K down projections and head, the 128-expert layer of Qwen3-30B-A3B), with
fewer layers where a whole model would only repeat them.  Weights are quantized blocks whose
values spread as trained ones do (standard deviation about 0.02, centred), norm weights lie
in [0.5, 1.5], activations and cache rows are N(0, 1).
"""
import hashlib
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skyla-kernel_amd"))

from skyla_hip import engine as E  # noqa: E402
from skyla_hip.abi import Context  # noqa: E402

PRECISIONS = ("f16", "q8", "f16_keys_q8_values")
EPS = 1e-6
THETA = 1e6
HEAD = 128
TYPES = {"q8_0": E.DType.Q8_0, "q4k": E.DType.Q4K, "q6k": E.DType.Q6K}
BLOCK = {"q8_0": (32, 34), "q4k": (256, 144), "q6k": (256, 210)}


def listed():
    small = {"n_embd": 1024, "n_head": 16, "n_kv": 8, "n_ff": 3072, "quant": "q8_0"}
    large = {"n_embd": 4096, "n_head": 32, "n_kv": 8, "n_ff": 12288, "quant": "q4k"}
    moe = {"n_embd": 2048, "n_ff": 768, "n_expert": 128, "n_used": 8}
    return [
        # one token's products through six layers of Qwen3-0.6B: small launches, where
        # latency counts more than bytes
        {"name": "matvecs-0.6b-q8", "kind": "matvecs", "layers": 6, **small},
        # one token's products through four layers of Qwen3-8B: the weights stream from HBM
        {"name": "matvecs-8b-q4k", "kind": "matvecs", "layers": 4, **large},
        # a ragged prompt tail through one layer of Qwen3-0.6B
        {"name": "matmuls-0.6b-q8-m200", "kind": "matmuls", "tokens": 200, **small},
        # a short prompt through one layer of Qwen3-8B
        {"name": "matmuls-8b-q4k-m37", "kind": "matmuls", "tokens": 37, **large},
        # a batch of 512 token rows through one layer of Qwen3-8B: the matrix cores' case
        {"name": "matmuls-8b-q4k-m512", "kind": "matmuls", "tokens": 512, **large},
        # one decode token through two 128-expert layers, eight experts each
        {"name": "moe-decode", "kind": "moe", "tokens": 1, "layers": 2, **moe},
        # a ragged prompt tail and a full prefill chunk through such a layer
        {"name": "moe-prefill-45", "kind": "moe", "tokens": 45, "layers": 1, **moe},
        {"name": "moe-prefill-128", "kind": "moe", "tokens": 128, "layers": 1, **moe},
        # a chat turn's next token in Qwen3-0.6B, the whole model with its tied head
        {"name": "step-0.6b", "kind": "step", "layers": 28, "n_vocab": 151936, "pos": 40,
         "kv": "f16_keys_q8_values", **small},
        # the next token after a long document, four layers of Qwen3-8B
        {"name": "step-8b-16k", "kind": "step", "layers": 4, "n_vocab": 8192, "pos": 16384,
         "kv": "f16_keys_q8_values", **large},
        # a chat prompt of 60 tokens into Qwen3-0.6B, four layers, f16 cache
        {"name": "prefill-0.6b-60", "kind": "prefill", "layers": 4, "n_vocab": 8192, "pos": 0, "tokens": 60,
         "kv": "f16", **small},
        # a 512-token prompt into Qwen3-8B, four layers
        {"name": "prefill-8b-512", "kind": "prefill", "layers": 4, "n_vocab": 8192, "pos": 0, "tokens": 512,
         "kv": "f16_keys_q8_values", **large},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng):
    """A dense layer's sizes: Q8_0 rows of any multiple of 32 values, Q4_K of 256."""
    quant = rng.choice(("q8_0", "q4k"))
    unit = 32 if quant == "q8_0" else 256
    n_kv = rng.choice((1, 2, 4, 8))
    rep = rng.choice((1, 2, 4, 8))
    while n_kv * rep > 32:
        rep //= 2
    n_embd = max(256, _log(rng, 512, 4096) // unit * unit)
    n_ff = max(256, _log(rng, 1024, 12288) // unit * unit)
    return {"n_embd": n_embd, "n_head": n_kv * rep, "n_kv": n_kv, "n_ff": n_ff, "quant": quant}


def draw(rng):
    kind = rng.choice(("matvecs", "matmuls", "moe", "step", "prefill"))
    if kind == "matvecs":
        return {"kind": kind, "layers": rng.randint(1, 4), **_shape(rng)}
    if kind == "matmuls":
        return {"kind": kind, "tokens": _log(rng, 2, 512), **_shape(rng)}
    if kind == "moe":
        n_expert = rng.choice((16, 48, 64, 128))
        return {"kind": kind, "tokens": rng.choice((1, _log(rng, 2, 128))), "layers": 1,
                "n_embd": 256 * rng.randint(2, 8), "n_ff": 256 * rng.randint(1, 3), "n_expert": n_expert,
                "n_used": rng.choice((2, 4, 8))}
    more = {"kind": kind, "layers": rng.randint(1, 4), "n_vocab": 64 * rng.randint(16, 128),
            "kv": rng.choice(PRECISIONS), **_shape(rng)}
    if kind == "step":
        return {**more, "pos": _log(rng, 1, 16384)}
    return {**more, "tokens": _log(rng, 2, 512), "pos": rng.choice((0, 0, _log(rng, 1, 2048)))}


# ---- inputs -----------------------------------------------------------------------------------
def _seed(seed, name):
    return int.from_bytes(hashlib.sha256(f"{seed}/{name}".encode()).digest()[:8], "little") >> 1


class Source:
    """Seeded inputs on the GPU, each tensor from its own name."""

    def __init__(self, seed):
        self.seed = seed

    def _gen(self, name):
        return torch.Generator("cuda").manual_seed(_seed(self.seed, name))

    def normal(self, name, *shape):
        return torch.randn(*shape, generator=self._gen(name), device="cuda")

    def uniform(self, name, lo, hi, *shape):
        return torch.rand(*shape, generator=self._gen(name), device="cuda") * (hi - lo) + lo

    def integers(self, name, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self._gen(name), device="cuda")

    def blocks(self, name, quant, n_in, n_rows):
        """Raw GGUF blocks of an [n_rows] x n_in matrix, (blocks, block bytes) uint8: uniform
        quants, scales such that the values have a standard deviation near 0.02, and for Q4_K
        minimums that centre each sub-block."""
        per, size = BLOCK[quant]
        n, g = n_rows * (n_in // per), self._gen(name)

        def half(lo, hi):
            v = torch.rand(n, generator=g, device="cuda") * (hi - lo) + lo
            return v.to(torch.float16).view(torch.uint8).view(n, 2)

        b = torch.randint(0, 256, (n, size), dtype=torch.uint8, generator=g, device="cuda")
        if quant == "q4k":
            d = torch.rand(n, generator=g, device="cuda") * 2e-4 + 6.5e-5
            b[:, 0:2] = d.to(torch.float16).view(torch.uint8).view(n, 2)
            b[:, 2:4] = (7.5 * d).to(torch.float16).view(torch.uint8).view(n, 2)
            # the 6-bit minimums equal the scales: bytes 4..7 = 0..3's, and in 8..11 the high
            # nibbles (minimums 4..7) the low ones (scales 4..7)
            b[:, 8:12] = b[:, 4:8]
            b[:, 12:16] = (b[:, 12:16] & 15) * 17
        elif quant == "q6k":
            b[:, 192:208] = torch.randint(-64, 65, (n, 16), dtype=torch.int8, generator=g, device="cuda").view(torch.uint8)
            b[:, 208:210] = half(1.5e-5, 4.5e-5)
        else:
            b[:, 0:2] = half(1e-4, 4.5e-4)
            b[:, 2:34] = torch.randint(-127, 128, (n, 32), dtype=torch.int8, generator=g, device="cuda").view(torch.uint8)
        return b


def _layer_mats(case, layer):
    """(name, type, n_in, n_out, accumulates) of a dense layer's matrices."""
    e, q, kv, ff = case["n_embd"], case["n_head"] * HEAD, case["n_kv"] * HEAD, case["n_ff"]
    t = case["quant"]
    down = "q6k" if t == "q4k" and layer % 2 == 0 else t
    return [("q", t, e, q, False), ("k", t, e, kv, False), ("v", t, e, kv, False), ("o", t, q, e, True),
            ("gate", t, e, ff, False), ("up", t, e, ff, False), ("down", down, ff, e, True)]


STAGES = (("q", "k", "v"), ("o",), ("gate", "up"), ("down",))
READS = {"q": "n", "k": "n", "v": "n", "o": "attn", "gate": "n", "up": "n", "down": "h"}
WRITES = {"q": "q", "k": "k", "v": "v", "o": "x", "gate": "gate", "up": "up", "down": "x"}


def _widths(case):
    return {"n": case["n_embd"], "attn": case["n_head"] * HEAD, "h": case["n_ff"], "x": case["n_embd"],
            "q": case["n_head"] * HEAD, "k": case["n_kv"] * HEAD, "v": case["n_kv"] * HEAD, "gate": case["n_ff"],
            "up": case["n_ff"]}


# ---- states -----------------------------------------------------------------------------------
_context = None


def _ctx():
    global _context
    if _context is None:
        _context = Context.new(0)
        # Context.new's symbol lookups leave HIP's last error set, which torch would report at
        # its next launch as its own; creating a pipeline clears it
        _context.create_pipeline("take_last", 2, 16, []).free()
    return _context


class _Owner:
    """Frees what a state holds on the GPU once nothing refers to it (its outputs do)."""

    def __init__(self):
        self.recordings, self.buffers, self.engine = [], [], None

    def __del__(self):
        for r in self.recordings:
            r.free()
        for b in self.buffers:
            b.free()
        if self.engine is not None:
            self.engine.free()


class _Memory:
    def __init__(self, owner, ptr, n, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False), "version": 3,
                                         "strides": None}


def _view(owner, buffer, kind="<f4", first=0, count=None):
    """A buffer's device memory as a flat tensor, elements [first, first + count)."""
    size = np.dtype(kind).itemsize
    if count is None:
        count = buffer.size // size - first
    return torch.as_tensor(_Memory(owner, buffer.device_ptr() + first * size, count, kind), device="cuda")


def _rows(flat, off, stride, rows, width):
    return flat[off: off + stride * rows].view(rows, stride)[:, :width] if rows > 1 else flat[off: off + width].view(1, width)


def _host(blocks):
    return blocks.reshape(-1).cpu().numpy()


class _State:
    pass


def _prepare_layers(case, seed):
    """matvecs and matmuls: weights laid out by the planner, an arena of activation rows and
    a recording of the products, as skyla-engine's graph records them."""
    ctx, src, owner, st = _ctx(), Source(seed), _Owner(), _State()
    decode = case["kind"] == "matvecs"
    layers, tokens = case.get("layers", 1), case.get("tokens", 1)
    plan = E.Planner(ctx.max_buffer())
    mats = []
    for i in range(layers):
        mats.append({name: plan.matrix(TYPES[t], n_in, n_out, _host(src.blocks(f"{i}.{name}", t, n_in, n_out)))
                     for name, t, n_in, n_out, _ in _layer_mats(case, i)})
    weights = E.upload_weights(ctx, plan)
    width, off, size = _widths(case), {}, 64
    for i in range(layers):
        for name, w in width.items():
            stride = -(-w // 64) * 64
            off[i, name] = (size, stride)
            size += stride * tokens
    arena = ctx.alloc_host((size + 64) * 4)
    owner.buffers = weights + [arena]
    flat = _view(owner, arena)
    for (i, name), (o, stride) in off.items():
        if name in ("n", "attn", "h", "x"):
            _rows(flat, o, stride, tokens, width[name]).copy_(src.normal(f"{i}.in.{name}", tokens, width[name]))
    _view(owner, arena, "<i4")[2] = tokens
    kernels = E.Kernels(ctx, weights, arena)
    tiles = -(-tokens // E.MATMUL_TILE_COLS)

    def body(r):
        g = E.Graph(r, kernels, None, None, not decode)
        for i in range(layers):
            for stage in STAGES:
                for name in stage:
                    x, y = off[i, READS[name]], off[i, WRITES[name]]
                    g.matvec(mats[i][name], x, y, name in ("o", "down"), not decode, groups_z=tiles)
                g.r.barrier()
        r.host_barrier()

    torch.cuda.synchronize()
    recording = ctx.record(False, body)
    owner.recordings = [recording]
    st.run = lambda: ctx.replay(recording)
    st.out = [{name: _rows(flat, *off[i, name], tokens, width[name]) for name in ("q", "k", "v", "x", "gate", "up")}
              for i in range(layers)]
    return st


def _moe_config(case):
    return E.Config(n_embd=case["n_embd"], n_ff=64, n_expert=case["n_expert"], n_expert_used=case["n_used"],
                    n_ff_expert=case["n_ff"])


def _moe_inputs(case, src):
    e, ff, n = case["n_embd"], case["n_ff"], case["n_expert"]
    for i in range(case["layers"]):
        yield (src.normal(f"{i}.router", n, e) * 0.02,
               [(name, n_in, n_out, src.blocks(f"{i}.{name}", "q4k", n_in, n * n_out))
                for name, n_in, n_out in (("gate", e, ff), ("up", e, ff), ("down", ff, e))])


def _prepare_moe(case, seed):
    """A stack of MoE layers on the same normed rows, each adding to the residual rows."""
    ctx, src, owner, st = _ctx(), Source(seed), _Owner(), _State()
    c, tokens = _moe_config(case), case["tokens"]
    plan, layers = E.Planner(ctx.max_buffer()), []
    for router, mats in _moe_inputs(case, src):
        layers.append([plan.matrix(TYPES["q4k"], n_in, n_out, _host(b)) for _, n_in, n_out, b in mats]
                      + [plan.table(router.cpu().numpy())])
    weights = E.upload_weights(ctx, plan)
    a = E.Arena(ctx, c)
    owner.buffers = weights + [a.buffer]
    flat, words = _view(owner, a.buffer), _view(owner, a.buffer, "<i4")
    _rows(flat, a.n, a.s_embd, tokens, c.n_embd).copy_(src.normal("n", tokens, c.n_embd))
    _rows(flat, a.x, a.s_embd, tokens, c.n_embd).copy_(src.normal("x", tokens, c.n_embd))
    words[2] = tokens
    kernels = E.Kernels(ctx, weights, a.buffer)

    def body(r):
        for gate, up, down, router in layers:
            E.Graph(r, kernels, a, c, tokens > 1).moe(gate, up, down, router)
        r.host_barrier()

    torch.cuda.synchronize()
    recording = ctx.record(False, body)
    owner.recordings = [recording]
    st.run = lambda: ctx.replay(recording)
    slots = tokens * case["n_used"]
    st.out = {"x": _rows(flat, a.x, a.s_embd, tokens, c.n_embd), "experts": words[a.moe.ids: a.moe.ids + slots],
              "weights": flat[a.moe.weights: a.moe.weights + slots]}
    return st


def _model_config(case):
    return E.Config(n_embd=case["n_embd"], n_ff=case["n_ff"], n_head=case["n_head"], n_head_kv=case["n_kv"],
                    head_dim=HEAD, n_vocab=case["n_vocab"], n_layer=case["layers"], eps=EPS, rope_theta=THETA)


def _model(case, src):
    """The tensors of a Qwen3 model by their GGUF names: f32 vectors on the GPU, and for
    matrices (type, n_in, n_out, blocks)."""
    e, v = case["n_embd"], case["n_vocab"]
    t = {"token_embd.weight": (case["quant"], e, v, src.blocks("embd", case["quant"], e, v)),
         "output_norm.weight": src.uniform("out_norm", 0.5, 1.5, e)}
    if case["quant"] == "q4k":  # Q8_0 models tie the head to the embedding
        t["output.weight"] = ("q6k", e, v, src.blocks("output", "q6k", e, v))
    names = {"q": "attn_q", "k": "attn_k", "v": "attn_v", "o": "attn_output", "gate": "ffn_gate", "up": "ffn_up",
             "down": "ffn_down"}
    for i in range(case["layers"]):
        for norm, n in (("attn_norm", e), ("ffn_norm", e), ("attn_q_norm", HEAD), ("attn_k_norm", HEAD)):
            t[f"blk.{i}.{norm}.weight"] = src.uniform(f"{i}.{norm}", 0.5, 1.5, n)
        for name, ty, n_in, n_out, _ in _layer_mats(case, i):
            t[f"blk.{i}.{names[name]}.weight"] = (ty, n_in, n_out, src.blocks(f"{i}.{name}", ty, n_in, n_out))
    return t


def _tokens(case, src):
    return [int(v) for v in src.integers("tokens", 0, case["n_vocab"], case.get("tokens", 1)).cpu()]


def _max_ctx(case):
    return case["pos"] + case.get("tokens", 1) + 8


def _stored(rows, q8):
    """Cache rows as they are stored: f16, or per 32 values one f16 scale and 8-bit quants."""
    if not q8:
        return rows.to(torch.float16), None
    y = rows.reshape(rows.numel() // 32, 32)
    s = (y.abs().amax(1) / 127.0).to(torch.float32)
    q = torch.round(torch.where(s[:, None] > 0, y / s[:, None], torch.zeros_like(y))).clamp(-127, 127)
    return q.to(torch.int8).reshape(rows.shape), s.to(torch.float16).reshape(rows.shape[0], rows.shape[1] // 32)


def _read(rows, scales):
    if scales is None:
        return rows.double()
    return (rows.double().reshape(*scales.shape, 32) * scales.double()[..., None]).reshape(rows.shape)


def _cache(case, src, layer, what):
    """The rows ("keys" or "values") already in a layer's cache, as stored."""
    pr = E.KvPrecision[case["kv"].upper()]
    rows = src.normal(f"{layer}.{what}", case["pos"], case["n_kv"] * HEAD)
    return _stored(rows, pr.keys_q8 if what == "keys" else pr.values_q8)


def _prepare_engine(case, seed):
    ctx, src, owner, st = _ctx(), Source(seed), _Owner(), _State()
    c, pr = _model_config(case), E.KvPrecision[case["kv"].upper()]
    tensors = {}
    for k, v in _model(case, src).items():
        tensors[k] = (TYPES[v[0]], v[1], v[2], _host(v[3])) if isinstance(v, tuple) else v.cpu().numpy()
    eng = owner.engine = E.Engine(ctx, tensors, c, _max_ctx(case), pr)
    a, kv = eng.arena, eng.arena.kv_layout
    first, tokens, dim = case["pos"], _tokens(case, src), c.n_head_kv * c.head_dim
    last = len(tokens) - (len(tokens) - 1) // E.BATCH * E.BATCH  # rows of the last chunk
    st.out = {"x": _rows(_view(owner, a.buffer), a.x, a.s_embd, last, c.n_embd)}
    half, byte = _view(owner, a.kv, "<f2"), _view(owner, a.kv, "|i1")
    for what, q8, off, scale_off in (("keys", pr.keys_q8, kv.keys(0), kv.key_scales(0)),
                                     ("values", pr.values_q8, kv.values(0), kv.value_scales(0))):
        regions = [(what, byte if q8 else half, off, dim)] + ([(what + " scales", half, scale_off, dim // 32)] if q8 else [])
        for i, (name, flat, o, width) in enumerate(regions):
            cache = flat[o: o + c.n_layer * a.max_ctx * width].view(c.n_layer, a.max_ctx, width)
            for l in range(c.n_layer):
                cache[l, :first] = _cache(case, src, l, what)[i]
            # 8-bit rows of a prompt are not compared one by one: the f16 products' rounding
            # moves some of them by a step (their scales and what attends to them are)
            if not (q8 and i == 0 and case["kind"] == "prefill"):
                st.out[name] = cache[:, first: first + len(tokens)]
    torch.cuda.synchronize()
    # a program that serves requests has recorded the graphs of these positions
    if case["kind"] == "step":
        eng.recording(False, first + 1)
    else:
        for at in range(0, len(tokens), E.BATCH):
            eng.recording(True, first + at + E.BATCH)

    def step():
        eng.pos = first
        st.out["logits"] = eng.step(tokens[0])

    def prefill():
        eng.pos = first
        st.out["logits"] = eng.prefill(tokens)

    st.run = step if case["kind"] == "step" else prefill
    return st


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("matvecs", "matmuls"):
        return _prepare_layers(case, seed)
    return _prepare_moe(case, seed) if kind == "moe" else _prepare_engine(case, seed)


def run(state):
    state.run()
    return state.out


# ---- what a pass cannot do without ------------------------------------------------------------
def _row_bytes(t, n):
    return n // BLOCK[t][0] * BLOCK[t][1]


def work(case):
    kind, m = case["kind"], case.get("tokens", 1)
    if kind == "moe":
        e, ff, n, used = case["n_embd"], case["n_ff"], case["n_expert"], case["n_used"]
        expert = 2 * ff * _row_bytes("q4k", e) + e * _row_bytes("q4k", ff)
        hit = n * (1 - (1 - used / n) ** m)  # experts that some token selects, on average
        nbytes = case["layers"] * (hit * expert + 4 * n * e + 4 * m * e * 3 + 8 * m * used)
        return {"bytes": nbytes, "flops": case["layers"] * 2.0 * m * (used * 3 * e * ff + n * e)}
    nbytes, flops = 0.0, 0.0
    for i in range(case.get("layers", 1)):
        for name, t, n_in, n_out, accum in _layer_mats(case, i):
            nbytes += n_out * _row_bytes(t, n_in)
            flops += 2.0 * m * n_in * n_out
            if kind in ("matvecs", "matmuls"):
                nbytes += 4 * m * n_out * (2 if accum else 1)
        if kind in ("matvecs", "matmuls"):
            nbytes += 4 * m * sum(_widths(case)[w] for w in ("n", "attn", "h"))
    if kind in ("matvecs", "matmuls"):
        return {"bytes": nbytes, "flops": flops}
    pr = E.KvPrecision[case["kv"].upper()]
    e, v, pos, dim = case["n_embd"], case["n_vocab"], case["pos"], case["n_kv"] * HEAD
    per = sum(dim + dim // 16 if q8 else 2 * dim for q8 in (pr.keys_q8, pr.values_q8))
    head = "q6k" if case["quant"] == "q4k" else case["quant"]
    nbytes += case["layers"] * (pos + m) * per + v * _row_bytes(head, e) + m * _row_bytes(case["quant"], e) + 4 * v
    seen = m * pos + m * (m + 1) / 2  # (query, position) pairs
    flops += 2.0 * v * e + case["layers"] * 4.0 * seen * case["n_head"] * HEAD
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """One token: f32 products and sums in another order differ by 1.5e-7, through layers and a
    16k-position cache (stored in 16 and 8 bits) the logits by 1e-4 from their 64-bit values.
    Token rows: f16 operands with f32 sums lie 6e-4 from the 64-bit products, and through the
    layers of a prompt such roundings grow to 8e-3 of the logits."""
    kind = case["kind"]
    if kind == "matvecs" or (kind == "moe" and case["tokens"] == 1):
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "step":
        return {"rel": 1e-3, "max": 2e-2, "differ": 0.005}
    if kind == "prefill":
        return {"rel": 0.025, "max": 0.3}
    return {"rel": 2.5e-3, "max": 2e-2}


# ---- the same in 64 bits ----------------------------------------------------------------------
def _values(t, blocks, n_in):
    """The f64 values of raw blocks, (rows, n_in)."""
    b = blocks.to(torch.int32)
    half = lambda i: blocks[:, i: i + 2].contiguous().view(torch.float16).double()  # noqa: E731
    n = blocks.shape[0]
    if t == "q8_0":
        w = half(0) * blocks[:, 2:34].contiguous().view(torch.int8).double()
    elif t == "q4k":
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:144].view(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(n, 8, 32).double()
        w = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    else:
        ql, qh = b[:, 0:128].view(n, 2, 64), b[:, 128:192].view(n, 2, 32)
        low = torch.stack([ql[:, :, :32] & 15, ql[:, :, 32:] & 15, ql[:, :, :32] >> 4, ql[:, :, 32:] >> 4], 2)
        high = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        q = (low | (high << 4)).reshape(n, 16, 16).double() - 32
        sc = blocks[:, 192:208].contiguous().view(torch.int8).double()
        w = half(208) * (sc[:, :, None] * q).reshape(n, 256)
    return w.reshape(-1, n_in)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _silu(v):
    return v / (1 + torch.exp(-v))


def _exact_layers(case, seed):
    src, m, width, out = Source(seed), case.get("tokens", 1), _widths(case), []
    for i in range(case.get("layers", 1)):
        v = {n: src.normal(f"{i}.in.{n}", m, width[n]).double() for n in ("n", "attn", "h", "x")}
        for name, t, n_in, n_out, accum in _layer_mats(case, i):
            y = v[READS[name]] @ _values(t, src.blocks(f"{i}.{name}", t, n_in, n_out), n_in).T
            v[WRITES[name]] = v[WRITES[name]] + y if accum else y
        out.append({n: v[n] for n in ("q", "k", "v", "x", "gate", "up")})
    return out


def _exact_moe(case, seed):
    src, m, used = Source(seed), case["tokens"], case["n_used"]
    n, x = src.normal("n", m, case["n_embd"]).double(), src.normal("x", m, case["n_embd"]).double()
    for router, mats in _moe_inputs(case, src):
        w = {name: _values("q4k", b, n_in).view(case["n_expert"], n_out, n_in) for name, n_in, n_out, b in mats}
        top, ids = torch.sort(n @ router.double().T, dim=1, descending=True, stable=True)
        weights, ids = torch.softmax(top[:, :used], 1), ids[:, :used]
        for t in range(m):
            for s in range(used):
                e = ids[t, s]
                h = _silu(w["gate"][e] @ n[t]) * (w["up"][e] @ n[t])
                x[t] += weights[t, s] * (w["down"][e] @ h)
    return {"x": x, "experts": None, "weights": weights.reshape(-1)}


def _rope(x, pos):
    freq = THETA ** (-2.0 * torch.arange(HEAD // 2, device="cuda", dtype=torch.float64) / HEAD)
    a = pos.double()[:, None, None] * freq
    lo, hi = x[..., : HEAD // 2], x[..., HEAD // 2:]
    return torch.cat([lo * torch.cos(a) - hi * torch.sin(a), lo * torch.sin(a) + hi * torch.cos(a)], -1)


def _exact_engine(case, seed):
    src = Source(seed)
    t, tokens, first = _model(case, src), _tokens(case, src), case["pos"]
    pr, m = E.KvPrecision[case["kv"].upper()], case.get("tokens", 1)
    n_head, n_kv = case["n_head"], case["n_kv"]
    w = lambda name: _values(t[name][0], t[name][3], t[name][1])  # noqa: E731
    ty, e, _, blocks = t["token_embd.weight"]
    per = e // BLOCK[ty][0]
    rows = blocks.view(-1, per, BLOCK[ty][1])[torch.tensor(tokens, device="cuda")]
    x = _values(ty, rows.reshape(-1, BLOCK[ty][1]), e)
    pos = torch.arange(first, first + m, device="cuda")
    last = m - (m - 1) // E.BATCH * E.BATCH
    out = {}
    for what, q8 in (("keys", pr.keys_q8), ("values", pr.values_q8)):
        out[what + " scales" if q8 else what] = []
        if q8 and case["kind"] == "step":
            out[what] = None
    for l in range(case["layers"]):
        p = lambda s: f"blk.{l}.{s}.weight"  # noqa: E731
        n = _norm(x, t[p("attn_norm")])
        q = _rope(_norm((n @ w(p("attn_q")).T).view(m, n_head, HEAD), t[p("attn_q_norm")]), pos)
        k = _rope(_norm((n @ w(p("attn_k")).T).view(m, n_kv, HEAD), t[p("attn_k_norm")]), pos).reshape(m, -1)
        v = n @ w(p("attn_v")).T
        cached = []
        for what, new, q8 in (("keys", k, pr.keys_q8), ("values", v, pr.values_q8)):
            out[what + " scales" if q8 else what].append(new.reshape(m, -1, 32).abs().amax(2) / 127.0 if q8 else new)
            rows = torch.cat([_read(*_cache(case, src, l, what)), _read(*_stored(new, q8))])
            cached.append(rows.view(first + m, n_kv, HEAD))
        keys, values = cached
        seen = torch.arange(first + m, device="cuda")[None, :] <= pos[:, None]
        att = []
        for h in range(n_head):
            s = (q[:, h] @ keys[:, h // (n_head // n_kv)].T) / math.sqrt(HEAD)
            att.append(torch.softmax(s.masked_fill(~seen, -math.inf), 1) @ values[:, h // (n_head // n_kv)])
        x = x + torch.cat(att, 1) @ w(p("attn_output")).T
        n = _norm(x, t[p("ffn_norm")])
        x = x + (_silu(n @ w(p("ffn_gate")).T) * (n @ w(p("ffn_up")).T)) @ w(p("ffn_down")).T
    out = {k: v if v is None else torch.stack(v) for k, v in out.items()}
    out["x"] = x[m - last:]
    head = w("output.weight" if "output.weight" in t else "token_embd.weight")
    out["logits"] = head @ _norm(x[-1], t["output_norm.weight"])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("matvecs", "matmuls"):
        return _exact_layers(case, seed)
    return _exact_moe(case, seed) if kind == "moe" else _exact_engine(case, seed)
