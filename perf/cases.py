"""The work this framework is measured on: calls of its public entry points (marmot_amd.HipBackend and the C ABI of
include/marmot_hip.h) at the sizes inference runs them at, on weights in native GGUF blocks.

Operations of a case ("op"):
  linear     marmot_hip_matmul_quantized: `tokens` rows of `dtype` activations against one [m, k] weight of `kind`.
             layers == 1: one eager call. layers > 1: the same linear of that many layers, one after the other, each with
             weights, input and output of its own, submitted as one HIP graph, the way a decode loop submits its steps.
  layer      one decoder layer from hidden states to hidden states: norm, q / k / v, rotary embedding, paged attention,
             o, residual, norm, gate / up, SwiGLU, down, residual; Q4_K weights with Q6_K for v and down.
  attention  marmot_hip_paged_attention: `new` tokens of each of `sequences` sequences over about `history` cached ones.
  moe        marmot_hip_moe_experts: `tokens` rows routed to `top_k` of `experts` gated feed-forward experts.
`replay`: the pass is one replay of a captured HIP graph (a decode step), else it is a row of eager calls (a prompt).
"""
import ctypes as C
import math

import torch

from marmot_amd import HipBackend, capi, row_bytes

KINDS = {"q4_0": capi.KIND_Q4_0, "q8_0": capi.KIND_Q8_0, "q4_k": capi.KIND_Q4_K, "q5_k": capi.KIND_Q5_K,
         "q6_k": capi.KIND_Q6_K}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
DT = {"f32": capi.DT_F32, "f16": capi.DT_F16, "bf16": capi.DT_BF16}
BLOCK = 16  # positions per block of the paged KV cache
MOST_FLOPS = 5e11  # of a drawn case: below the largest listed one


def linear(name, kind, tokens, k, m, dtype="f32", bias=False, layers=1):
    return {"name": name, "op": "linear", "kind": kind, "tokens": tokens, "k": k, "m": m, "dtype": dtype, "bias": bias,
            "layers": layers}


def layer(name, sequences, new, history, cache, replay):
    return {"name": name, "op": "layer", "sequences": sequences, "new": new, "history": history, "cache": cache,
            "hidden": 4096, "ffn": 14336, "heads": 32, "kv_heads": 8, "head_dim": 128, "replay": replay}


def attention(name, sequences, new, history, heads, kv_heads, head_dim, act, cache):
    return {"name": name, "op": "attention", "sequences": sequences, "new": new, "history": history, "heads": heads,
            "kv_heads": kv_heads, "head_dim": head_dim, "act": act, "cache": cache}


def moe(name, tokens, kind, experts, top_k, hidden, ffn, replay):
    return {"name": name, "op": "moe", "tokens": tokens, "kind": kind, "experts": experts, "top_k": top_k,
            "hidden": hidden, "ffn": ffn, "replay": replay}


def listed():
    return [
        # the smallest call: one token through a feed-forward projection of a 1.1B model, called by itself
        linear("single_q8_0", "q8_0", 1, 2048, 5632),
        # one token of one user: the down projections of eight layers of an 8B model, in one submission
        linear("decode_q4_k", "q4_k", 1, 14336, 4096, layers=8),
        # eight users decoding together, the wider format a Q4_K_M file keeps for the down projection
        linear("decode_q6_k_8", "q6_k", 8, 14336, 4096, layers=4),
        # the projection to the vocabulary at the end of every step
        linear("logits_q6_k", "q6_k", 1, 4096, 128256),
        # prompt with FLOAT16 activations (attention projection of an 8B model)
        linear("prompt_q4_k_f16", "q4_k", 512, 4096, 4096, dtype="f16"),
        # prompt of an uneven length with FLOAT32 activations (up projection)
        linear("prompt_q4_k", "q4_k", 1000, 4096, 14336),
        # short prompt, a format with 32-value blocks, with bias
        linear("prompt_q8_0", "q8_0", 300, 4096, 4096, bias=True),
        # a whole decoder layer, 16 users with about 4096 tokens of context each
        layer("layer_decode", 16, 1, 4095, "f16", True),
        # the same layer for a fresh prompt of one user
        layer("layer_prompt", 1, 1024, 0, "f16", False),
        # chunked prefill: two users' next 512 tokens over the 2048 that are cached already
        attention("attention_chunk", 2, 512, 2048, 32, 8, 128, "f32", "bf16"),
        # routed experts (128 of 768 over 2048 hidden, eight per token): a decode step of many users
        moe("moe_decode", 64, "q4_k", 128, 8, 2048, 768, True),
        # the same experts for prompts
        moe("moe_prompt", 2048, "q4_k", 128, 8, 2048, 768, False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    c = _draw(rng)
    c.pop("name")
    return c


def _draw(rng):
    what = rng.choice(("decode", "decode", "prompt", "prompt", "layer_decode", "layer_prompt", "attention", "moe"))
    kind = rng.choice(("q4_k", "q4_k", "q6_k", "q5_k", "q8_0", "q4_0"))
    if what in ("decode", "prompt"):
        k, m = 256 * _log(rng, 4, 56), _log(rng, 512, 16384)
        if rng.random() < 0.5:
            m = max(512, m // 256 * 256)
        if what == "decode":
            return linear("", kind, rng.choice((1, 1, 2, 3, 4, 6, 8, 11, 16)), k, m, layers=rng.choice((1, 4, 8)))
        tokens = min(_log(rng, 17, 2048), int(MOST_FLOPS / (2.0 * k * m)))
        return linear("", kind, tokens, k, m, dtype=rng.choice(("f32", "f32", "f16")), bias=rng.random() < 0.3)
    if what == "layer_decode":
        return layer("", rng.choice((1, 2, 5, 8, 16)), 1, _log(rng, 100, 4095), rng.choice(("f16", "f16", "bf16")), True)
    if what == "layer_prompt":
        new, seqs = _log(rng, 40, 1000), rng.choice((1, 1, 2, 3))
        return layer("", seqs, max(16, new // seqs), rng.choice((0, 0, 0, 700)), rng.choice(("f16", "f16", "bf16")), False)
    if what == "attention":
        kv = rng.choice((4, 8))
        new, seqs = _log(rng, 32, 1500), rng.choice((1, 2, 4))
        return attention("", seqs, max(8, new // seqs), rng.choice((0, _log(rng, 64, 4096))), kv * rng.choice((1, 4, 7)), kv,
                         rng.choice((64, 128, 128)), rng.choice(("f32", "f16")), rng.choice(("f16", "bf16")))
    tokens = _log(rng, 8, 2048)
    return moe("", tokens, rng.choice(("q4_k", "q4_k", "q6_k", "q5_k")), rng.choice((32, 64, 128)), rng.choice((2, 4, 8)),
               256 * rng.choice((4, 8)), 256 * rng.choice((2, 3, 4)), tokens <= 64)


# ---------------------------------------------------------------- preparation

_hip = None


def _backend():
    global _hip
    if _hip is None:
        _hip = HipBackend(0)
    return _hip


class _Buf:
    """A torch tensor as the buffer argument of a HipBackend method."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


class _State:
    """Tensors, and the captured graph of a replayed pass."""

    def __init__(self):
        self.keep, self.graph, self.step, self.out = [], None, None, None

    def hold(self, t):
        b = _Buf(t.contiguous())
        self.keep.append(b)
        return b

    def __del__(self):
        if self.graph is not None and _hip is not None:
            _hip.graph_destroy(self.graph)


def _vp(b):
    return C.c_void_p(b.ptr)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _weights(g, kind, rows, k):
    """[rows, row_bytes] blocks of N(0, 0.02) weights, through the framework's own quantizers where it has one."""
    hip, out = _backend(), torch.empty(rows, row_bytes(KINDS[kind], k), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 27) // k)
    for r in range(0, rows, step):
        w = _randn(g, min(step, rows - r), k).mul_(0.02)
        dst = out[r:r + step]
        if kind == "q4_0":
            b = w.reshape(-1, 32)
            at = b.abs().argmax(1, keepdim=True)
            d = (b.gather(1, at) / -8.0).to(torch.float16)
            df = d.float()
            q = torch.where(df != 0, b / df, torch.zeros_like(b)).add_(8.5).clamp_(0, 15).to(torch.uint8)
            blocks = torch.cat([d.view(torch.uint8), q[:, :16] | (q[:, 16:] << 4)], 1)
            dst.copy_(blocks.reshape(dst.shape))
            continue
        torch.cuda.synchronize()
        if kind == "q8_0":
            capi.check(hip.lib.marmot_hip_quantize_activations(hip.dev, capi.KIND_Q8_0, C.c_void_p(w.data_ptr()),
                                                               capi.DT_F32, w.shape[0], k, C.c_void_p(dst.data_ptr())))
        else:
            capi.check(hip.lib.marmot_hip_quantize_weights(hip.dev, KINDS[kind], C.c_void_p(w.data_ptr()), w.shape[0], k,
                                                           C.c_void_p(dst.data_ptr())))
        hip.synchronize()
    return out


def _finish(s, replay):
    """Runs the pass once (workspaces reach their size) and captures it when the program replays it."""
    hip = _backend()
    torch.cuda.synchronize()
    s.step()
    hip.synchronize()
    if replay:
        s.graph = hip.graph_capture(s.step)
    return s


def prepare(case, seed):
    s, g = _State(), _gen(seed)
    {"linear": _prepare_linear, "layer": _prepare_layer, "attention": _prepare_attention, "moe": _prepare_moe}[case["op"]](
        case, s, g)
    return _finish(s, case.get("replay", case.get("layers", 1) > 1))


def _prepare_linear(c, s, g):
    hip, kind, dt = _backend(), KINDS[c["kind"]], c["dtype"]
    n, k, m = c["tokens"], c["k"], c["m"]
    args = []
    for _ in range(c["layers"]):
        w, x = s.hold(_weights(g, c["kind"], m, k)), s.hold(_randn(g, n, k, dtype=TORCH[dt]))
        b = s.hold(_randn(g, m)) if c["bias"] else None
        args.append((w, x, b, s.hold(torch.empty(n, m, device="cuda"))))

    def step():
        for w, x, b, out in args:
            hip.linear_d(kind, w, x, DT[dt], n, k, m, out, capi.DT_F32, d_bias=b)

    s.step, s.out = step, [a[3].t for a in args]


def _sequences(c):
    """Cached length of every sequence: uneven, the longest has `history` positions."""
    h = c["history"]
    return [h - (i * 37) % (h // 4 + 1) for i in range(c["sequences"])]


def _prepare_cache(c, s, g, act):
    """Token metadata, block table (blocks in shuffled order, as an allocator leaves them) and the filled cache."""
    hkv, d, lens = c["kv_heads"], c["head_dim"], _sequences(c)
    need = [-(-(h + c["new"]) // BLOCK) for h in lens]
    order = torch.randperm(sum(need), generator=g, device="cuda").cpu().tolist()
    table = torch.full((len(lens), max(need)), 0xFFFFFFFF, dtype=torch.int64)
    meta, at = [], 0
    for i, h in enumerate(lens):
        table[i, :need[i]] = torch.tensor(order[at:at + need[i]])
        at += need[i]
        meta += [(i, p, int(table[i, p // BLOCK]) * BLOCK + p % BLOCK, 0) for p in range(h, h + c["new"])]
    as_u32 = lambda t: t.to(torch.int64).to("cuda").to(torch.int32)  # noqa: E731  (the bits of uint32)
    shape = (sum(need), 1, hkv, BLOCK, d)
    kv = [s.hold(_randn(g, *shape, dtype=TORCH[c["cache"]])) for _ in range(2)]
    meta = torch.tensor(meta, dtype=torch.int64)
    d_meta, d_table = s.hold(as_u32(meta)), s.hold(as_u32(torch.where(table == 0xFFFFFFFF, -1, table)))
    p = capi.PagedAttention()
    p.token_count, p.layer_idx, p.num_q_heads, p.num_kv_heads = len(meta), 0, c["heads"], hkv
    p.head_dim, p.block_size, p.scale, p.act_dtype, p.kv_dtype = d, BLOCK, d ** -0.5, DT[act], DT[c["cache"]]
    p.d_token_meta, p.meta_stride = d_meta.ptr, (C.c_size_t * 2)(4, 1)
    p.q_stride, p.out_stride = ((C.c_size_t * 3)(c["heads"] * d, d, 1) for _ in range(2))
    p.k_stride, p.v_stride = ((C.c_size_t * 3)(hkv * d, d, 1) for _ in range(2))
    p.d_kv_k, p.d_kv_v = kv[0].ptr, kv[1].ptr
    p.kv_stride = (C.c_size_t * 5)(hkv * BLOCK * d, hkv * BLOCK * d, BLOCK * d, d, 1)
    p.kv_blocks, p.kv_layers = shape[0], 1
    p.d_block_table, p.table_stride = d_table.ptr, (C.c_size_t * 2)(table.shape[1], 1)
    p.max_seqs, p.max_blocks_per_seq = table.shape
    return p, meta[:, 1], [b.t for b in kv]


def _prepare_attention(c, s, g):
    hip, d, dt = _backend(), c["head_dim"], TORCH[c["act"]]
    p, pos, kv = _prepare_cache(c, s, g, c["act"])
    t = len(pos)
    q, k, v = (s.hold(_randn(g, t, h, d, dtype=dt)) for h in (c["heads"], c["kv_heads"], c["kv_heads"]))
    out = s.hold(torch.empty(t, c["heads"], d, dtype=dt, device="cuda"))
    p.d_q, p.d_k_new, p.d_v_new, p.d_out = q.ptr, k.ptr, v.ptr, out.ptr

    def step():
        capi.check(hip.lib.marmot_hip_paged_attention(hip.dev, C.byref(p), 0))

    s.step, s.out = step, [out.t] + kv


def _layer_shapes(c):
    H, F, q, kv = c["hidden"], c["ffn"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    return {"q": ("q4_k", q, H), "k": ("q4_k", kv, H), "v": ("q6_k", kv, H), "o": ("q4_k", H, q),
            "gate": ("q4_k", F, H), "up": ("q4_k", F, H), "down": ("q6_k", H, F)}


def _prepare_layer(c, s, g):
    hip = _backend()
    lib, dev, chk = hip.lib, hip.dev, capi.check
    H, F, hq, hkv, d = c["hidden"], c["ffn"], c["heads"], c["kv_heads"], c["head_dim"]
    shapes, Q4, Q6, F32 = _layer_shapes(c), capi.KIND_Q4_K, capi.KIND_Q6_K, capi.DT_F32
    w = {n: s.hold(_weights(g, kind, m, k)) for n, (kind, m, k) in shapes.items()}
    pa, pos, kv = _prepare_cache(c, s, g, "f32")
    T = len(pos)
    new = lambda cols: s.hold(torch.empty(T, cols, device="cuda"))  # noqa: E731
    x, n1, n2 = s.hold(_randn(g, T, H)), s.hold(1 + 0.1 * _randn(g, H)), s.hold(1 + 0.1 * _randn(g, H))
    h, q, k, v, att, o, x1, h2 = (new(n) for n in (H, hq * d, hkv * d, hkv * d, hq * d, H, H, H))
    gate, up, down, y = new(F), new(F), new(H), new(H)
    pack = {n: s.hold(torch.empty(hip.packed_activation_bytes(Q4, T, cols), dtype=torch.uint8, device="cuda"))
            for n, cols in (("h", H), ("att", hq * d), ("h2", H), ("act", F))}
    pa.d_q, pa.d_k_new, pa.d_v_new, pa.d_out = q.ptr, k.ptr, v.ptr, att.ptr
    freqs, scale, hd = hip.rope_frequencies(d, head_dim=d, theta=500000.0)
    d_f = s.hold(torch.from_numpy(freqs).to("cuda"))
    p32 = pos.to("cuda").to(torch.int32)
    rope = {}
    for n, heads in (("q", hq), ("k", hkv)):
        rope[n] = capi.Rope(s.hold(p32.repeat_interleave(heads)).ptr, capi.DT_I32, d_f.ptr, scale, hd, 0, 0, 0)

    def lin(n, packed, out):
        kind, m, cols = shapes[n]
        hip.linear_prepacked_d(KINDS[kind], w[n], packed, T, cols, m, out)

    def norm(src, weight, out, packed):
        chk(lib.marmot_hip_rms_norm_pack(dev, _vp(src), None, _vp(weight), 0.0, 1e-5, T, H, Q4, _vp(out), _vp(packed)))

    def step():
        norm(x, n1, h, pack["h"])
        lin("q", pack["h"], q)
        lin("k", pack["h"], k)
        lin("v", pack["h"], v)
        chk(lib.marmot_hip_rope(dev, _vp(q), F32, T * hq, d, d, d, C.byref(rope["q"]), _vp(q)))
        chk(lib.marmot_hip_rope(dev, _vp(k), F32, T * hkv, d, d, d, C.byref(rope["k"]), _vp(k)))
        chk(lib.marmot_hip_paged_attention(dev, C.byref(pa), 0))
        hip.pack_activations_d(Q4, att, F32, T, hq * d, pack["att"])
        lin("o", pack["att"], o)
        chk(lib.marmot_hip_add(dev, _vp(x), _vp(o), T * H, _vp(x1)))
        norm(x1, n2, h2, pack["h2"])
        lin("gate", pack["h2"], gate)
        lin("up", pack["h2"], up)
        chk(lib.marmot_hip_swiglu_pack(dev, _vp(gate), _vp(up), T, F, Q6, _vp(pack["act"])))
        lin("down", pack["act"], down)
        chk(lib.marmot_hip_add(dev, _vp(x1), _vp(down), T * H, _vp(y)))

    s.step, s.out = step, [y.t] + kv


def _prepare_moe(c, s, g):
    hip, kind = _backend(), KINDS[c["kind"]]
    T, E, k, H, F = (c[n] for n in ("tokens", "experts", "top_k", "hidden", "ffn"))
    gate, up = (s.hold(_weights(g, c["kind"], E * F, H)) for _ in range(2))
    down, x = s.hold(_weights(g, c["kind"], E * H, F)), s.hold(_randn(g, T, H))
    val, ids = torch.topk(_randn(g, T, E), k, dim=1)
    ids, wts = s.hold(ids.to(torch.int32)), s.hold(torch.softmax(val, 1))
    out = s.hold(torch.empty(T, H, device="cuda"))

    def step():
        hip.moe_experts_d(x, T, H, F, E, k, kind, kind, gate, up, down, ids, wts, out)

    s.step, s.out = step, [out.t]


# ---------------------------------------------------------------- a pass, what it needs, how exact it is


def run(state):
    if state.graph is not None:
        _backend().graph_launch(state.graph)
    else:
        state.step()
    return state.out


def _attention_work(c, act_bytes):
    hq, hkv, d, lens, new = c["heads"], c["kv_heads"], c["head_dim"], _sequences(c), c["new"]
    tokens = new * len(lens)
    rows = sum(h + new for h in lens)  # every cached row once, the new ones written once
    pairs = sum(new * h + new * (new + 1) // 2 for h in lens)
    return {"bytes": rows * hkv * d * 2 * 2 + tokens * hkv * d * 2 * (2 + act_bytes) + 2 * tokens * hq * d * act_bytes,
            "flops": 4.0 * pairs * hq * d}


def work(case):
    c = case
    if c["op"] == "linear":
        n, k, m, size = c["tokens"], c["k"], c["m"], 4 if c["dtype"] == "f32" else 2
        one = m * row_bytes(KINDS[c["kind"]], k) + n * k * size + n * m * 4 + (4 * m if c["bias"] else 0)
        return {"bytes": c["layers"] * one, "flops": c["layers"] * 2.0 * n * k * m}
    if c["op"] == "attention":
        return _attention_work(c, 4 if c["act"] == "f32" else 2)
    if c["op"] == "layer":
        # values between the operations need not reach memory: weights, cache rows, hidden states in and out
        t, a = c["new"] * c["sequences"], _attention_work(c, 0)
        weights = sum(m * row_bytes(KINDS[kind], k) for kind, m, k in _layer_shapes(c).values())
        return {"bytes": weights + a["bytes"] + 2 * t * c["hidden"] * 4,
                "flops": a["flops"] + sum(2.0 * t * m * k for _, m, k in _layer_shapes(c).values())}
    T, E, k, H, F = (c[n] for n in ("tokens", "experts", "top_k", "hidden", "ffn"))
    active = E * (1.0 - (1.0 - k / E) ** T)  # experts that some token chose, expected
    one = 2 * F * row_bytes(KINDS[c["kind"]], H) + H * row_bytes(KINDS[c["kind"]], F)
    return {"bytes": active * one + 2 * T * H * 4, "flops": 6.0 * T * k * H * F}


def tolerance(case):
    """About four times what two correct routes of the same operation differ by."""
    # exact integer block sums (or exact FLOAT16 operands) summed in FLOAT32 in another order: 1e-7 to 4e-7
    if case["op"] == "linear":
        return {"rel": 2e-6, "max": 2e-5}
    # FLOAT32 softmax and sums in another order: 5e-7; FLOAT16 outputs differ by one rounding where they fall on a tie
    if case["op"] == "attention":
        return {"rel": 2e-6, "max": 3e-5} if case["act"] == "f32" else {"rel": 1e-4, "max": 2e-3}
    # activations are quantized to 8 bits between the linears, where one unit in the last place upstream moves a code by a
    # step: 9e-5 (largest 5e-3) over one such point, 6e-3 (largest 0.044) over the three of a layer
    if case["op"] == "moe":
        return {"rel": 4e-4, "max": 2e-2}
    return {"rel": 2.5e-2, "max": 0.18}
