"""The calls whose speed this repository keeps track of: what programs that use the library have it
do, over the range of sizes, data types and options that they use, through the public Python API.

A case is a dict of plain values. `listed()` are the fixed cases, `draw(rng)` gives one more of the
same ranges, `prepare` makes what a program holds before the call (device tensors, plans), `run` is
one pass, `exact` the same outputs from float64 torch operations, `work` the bytes and operations a
pass cannot do without and `tolerance` how far two correct implementations may differ.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "flat-attention_amd"))
import flat_attention_amd as fa  # noqa: E402

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
STORAGE = {"f32": fa.DTYPE_F32, "f16": fa.DTYPE_F16, "bf16": fa.DTYPE_BF16}
THETA = 10000.0


def listed():
    return [
        # The smallest call in use: the reference's own MHA example, f32, latency-bound.
        {"name": "mha_f32_small", "kind": "mha", "dtype": "f32", "batch": 1, "heads": 2,
         "seq": 128, "dim": 64, "causal": True},
        # Full-size f32 MHA (encoder or decoder layer run in f32), causal.
        {"name": "mha_f32_causal", "kind": "mha", "dtype": "f32", "batch": 4, "heads": 16,
         "seq": 2048, "dim": 128, "causal": True},
        # The prefill of a batch of two long prompts: GQA with fused RoPE, prepared once.
        {"name": "prefill_bf16", "kind": "gqa", "dtype": "bf16", "batch": 2, "q_heads": 32,
         "kv_heads": 8, "seq": 4096, "dim": 128, "causal": True, "layout": "prepared",
         "precise": False},
        # The prefill of one short prompt straight from the projections' layout.
        {"name": "prefill_short_f16", "kind": "gqa", "dtype": "f16", "batch": 1, "q_heads": 8,
         "kv_heads": 2, "seq": 512, "dim": 128, "causal": True, "layout": "projection",
         "precise": False},
        # A bidirectional GQA layer of 64-wide heads at an odd length.
        {"name": "gqa_d64_odd_bf16", "kind": "gqa", "dtype": "bf16", "batch": 2, "q_heads": 16,
         "kv_heads": 4, "seq": 999, "dim": 64, "causal": False, "layout": "heads",
         "precise": False},
        # One step of a chunked prefill: 512 new tokens of 8 sequences go into the page pool
        # (RoPE on append), then attend over 2048 cached tokens and themselves.
        {"name": "chunk_paged_bf16", "kind": "chunk", "dtype": "bf16", "seqs": 8, "q_heads": 32,
         "kv_heads": 8, "dim": 128, "cached": 2048, "new": 512, "page": 16},
        # A padded serving batch: chunks of different lengths after different cached prefixes.
        {"name": "variable_bf16", "kind": "variable", "dtype": "bf16", "seqs": 4, "q_heads": 32,
         "kv_heads": 8, "dim": 128, "query": 700, "kv": 1500},
        # One decode step of a full serving batch over a shuffled page pool.
        {"name": "decode_paged_bf16", "kind": "decode", "dtype": "bf16", "seqs": 64,
         "q_heads": 32, "kv_heads": 8, "dim": 128, "low": 512, "high": 8192, "page": 16},
        # One decode step of a small batch whose lengths change every token: tables and work
        # lists go in with the call, which allocates nothing.
        {"name": "decode_step_f16", "kind": "step", "dtype": "f16", "seqs": 8, "q_heads": 32,
         "kv_heads": 8, "dim": 128, "low": 100, "high": 2000, "page": 16},
        # Single-sequence decode over a resident f32 cache, the reference's published shape.
        {"name": "decode_resident_f32", "kind": "resident", "dtype": "f32", "batch": 1,
         "q_heads": 16, "kv_heads": 4, "dim": 64, "capacity": 8192, "live": 8192},
        # Attention of one training step, forward then recompute backward, full size.
        {"name": "train_bf16", "kind": "train", "dtype": "bf16", "batch": 2, "q_heads": 32,
         "kv_heads": 8, "seq": 4096, "dim": 128, "causal": True},
        # The same in f32 (the reference's backward is f32) at a small model's size.
        {"name": "train_f32", "kind": "train", "dtype": "f32", "batch": 1, "q_heads": 8,
         "kv_heads": 2, "seq": 512, "dim": 64, "causal": True},
    ]


# ------------------------------------------------------------------------------- drawn cases

def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _heads(rng):
    return rng.choice([(8, 2), (16, 4), (32, 8), (32, 8), (8, 8), (12, 4), (6, 1)])


def _cost(case):
    """Operations, an f32 one counted as 16 (the ratio of the matrix rates)."""
    return work(case)["flops"] * (16 if case["dtype"] == "f32" else 1)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= most:
            return case


def _draw(rng):
    kind = rng.choice(["mha", "gqa", "gqa", "chunk", "variable", "decode", "step", "resident",
                       "train", "train"])
    half = rng.choice(["bf16", "bf16", "f16"])
    hq, hkv = _heads(rng)
    if kind == "mha":
        dtype = rng.choice(["f32", "f32", half])
        dim, heads, batch = rng.choice([32, 64, 80, 128]), rng.choice([1, 2, 4, 8, 16]), rng.randint(1, 4)
        return {"kind": kind, "dtype": dtype, "batch": batch, "heads": heads,
                "seq": _log(rng, 32, 2048), "dim": dim, "causal": rng.random() < 0.5}
    if kind == "gqa":
        dtype = rng.choice([half, half, half, "f32"])
        layout = rng.choice(["prepared", "heads", "projection"])
        return {"kind": kind, "dtype": dtype, "batch": rng.randint(1, 2), "q_heads": hq,
                "kv_heads": hkv, "seq": _log(rng, 64, 4096 if dtype != "f32" else 1024),
                "dim": rng.choice([64, 128, 128]), "causal": rng.random() < 0.75,
                "layout": layout,
                "precise": layout == "prepared" and dtype == "bf16" and rng.random() < 0.3}
    if kind == "chunk":
        return {"kind": kind, "dtype": half, "seqs": rng.randint(1, 8), "q_heads": hq,
                "kv_heads": hkv, "dim": rng.choice([64, 128, 128]),
                "cached": _log(rng, 16, 2048), "new": _log(rng, 16, 512),
                "page": rng.choice([16, 16, 32])}
    if kind == "variable":
        query = _log(rng, 16, 700)
        return {"kind": kind, "dtype": half, "seqs": rng.randint(2, 6), "q_heads": hq,
                "kv_heads": hkv, "dim": rng.choice([64, 128, 128]), "query": query,
                "kv": query + _log(rng, 16, 1400)}
    if kind in ("decode", "step"):
        high = _log(rng, 128, 8192 if kind == "decode" else 2048)
        return {"kind": kind, "dtype": rng.choice([half, half, half, "f32"]),
                "seqs": _log(rng, 1, 64 if kind == "decode" else 16), "q_heads": hq,
                "kv_heads": hkv, "dim": rng.choice([64, 128, 128]), "low": max(16, high // 16),
                "high": high, "page": rng.choice([16, 16, 32])}
    if kind == "resident":
        capacity = 16 * _log(rng, 16, 512)
        return {"kind": kind, "dtype": rng.choice(["f32", half]), "batch": rng.randint(1, 4),
                "q_heads": hq, "kv_heads": hkv, "dim": rng.choice([64, 128]),
                "capacity": capacity, "live": rng.randint(capacity // 2, capacity)}
    dtype = rng.choice([half, half, "f32"])
    return {"kind": kind, "dtype": dtype, "batch": rng.randint(1, 2), "q_heads": hq,
            "kv_heads": hkv, "seq": _log(rng, 64, 4096 if dtype != "f32" else 1024),
            "dim": rng.choice([64, 128]), "causal": rng.random() < 0.8}


# ------------------------------------------------------------------------------- lengths

def _lengths(case):
    """The live tokens of each sequence of a decode batch (the same for every seed)."""
    r = np.random.default_rng([case["seqs"], case["low"], case["high"]])
    return r.integers(case["low"], case["high"] + 1, case["seqs"]).astype(np.int32)


def _spans(case):
    """(active queries, active K/V rows) of each sequence of a padded batch: the first fills the
    padding, the last is a single new token, the others lie between."""
    r = np.random.default_rng([case["seqs"], case["query"], case["kv"]])
    spans = [(case["query"], case["kv"])]
    for _ in range(case["seqs"] - 2):
        q = int(r.integers(1, case["query"] + 1))
        spans.append((q, q + int(r.integers(0, case["kv"] - case["query"] + 1))))
    spans.append((1, 1 + int(r.integers(0, case["kv"] - case["query"] + 1))))
    return spans


# ------------------------------------------------------------------------------- state

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = fa.HipContext(0)
    return _context


def _normal(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(TORCH[dtype])


def _inputs(case, seed):
    """The tensors of a case, in the order that its kind uses them, and its numpy generator."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    r = np.random.default_rng(int(seed))
    kind, dt = case["kind"], case["dtype"]
    if kind == "mha":
        shape = (case["batch"], case["heads"], case["seq"], case["dim"])
        return [_normal(gen, shape, dt) for _ in range(3)], r
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["dim"]
    if kind in ("gqa", "train"):
        b, s = case["batch"], case["seq"]
        if case.get("layout") == "projection":
            shapes = [(b, s, hq, d), (b, s, hkv, d), (b, s, hkv, d)]
        else:
            shapes = [(b, hq, s, d), (b, hkv, s, d), (b, hkv, s, d)]
        if kind == "train":
            shapes.append(shapes[0])
        return [_normal(gen, x, dt) for x in shapes], r
    n = case.get("seqs", case.get("batch"))
    if kind == "variable":
        return [_normal(gen, (n, case["query"], hq, d), dt),
                _normal(gen, (n, case["kv"], hkv, d), dt),
                _normal(gen, (n, case["kv"], hkv, d), dt)], r
    if kind == "resident":
        return [_normal(gen, (n, hq, d), dt), _normal(gen, (n, case["capacity"], hkv, d), dt),
                _normal(gen, (n, case["capacity"], hkv, d), dt)], r
    page = case["page"]
    if kind == "chunk":
        lens = np.full(n, case["cached"] + case["new"], np.int32)
        rows = (n, case["new"])
    else:
        lens = _lengths(case)
        rows = (n,)
    pages = (lens + page - 1) // page
    total = int(pages.sum())
    order = r.permutation(total).astype(np.int32)
    table = np.zeros((n, int(pages.max())), np.int32)
    at = 0
    for i in range(n):
        table[i, :pages[i]] = order[at:at + pages[i]]
        at += pages[i]
    pools = [_normal(gen, (total, page, hkv, d), dt) for _ in range(2)]
    tensors = [_normal(gen, rows + (hq, d), dt)] + pools
    if kind == "chunk":
        tensors += [_normal(gen, rows + (hkv, d), dt) for _ in range(2)]
    return tensors + [table, lens, total], r


def _buffer(t):
    return fa.DeviceBuffer(_ctx(), t.numel() * t.element_size(), t.data_ptr(), owned=False)


class _State:
    pass


def _output(st, layout, o_shape, lse_shape, dtype):
    """The packed [O | LSE] buffer of a call and its two parts as tensors."""
    st.packed = torch.empty(layout.combined_bytes, dtype=torch.uint8, device="cuda")
    st.out = _buffer(st.packed)
    st.o = st.packed[:layout.output_bytes].view(TORCH[dtype]).view(o_shape)
    at = layout.lse_byte_offset
    st.lse = st.packed[at:at + 4 * layout.lse_elements].view(torch.float32).view(lse_shape)


def prepare(case, seed):
    ctx, st = _ctx(), _State()
    tensors, _ = _inputs(case, seed)
    kind, dtype = case["kind"], STORAGE[case["dtype"]]
    st.case, st.tensors = case, tensors
    st.config = fa.FlatAttentionConfig(case.get("causal", True))
    if kind == "mha":
        st.shape = fa.AttentionShape(case["batch"], case["heads"], case["seq"], case["dim"])
        st.op = fa.HipFlatAttention(ctx, dtype)
        st.bufs = [_buffer(t) for t in tensors]
        _output(st, st.op.layout(st.shape), tensors[0].shape, tensors[0].shape[:3], case["dtype"])
    elif kind in ("gqa", "train"):
        b, hq, hkv, s, d = (case[x] for x in ("batch", "q_heads", "kv_heads", "seq", "dim"))
        st.shape = fa.GroupedAttentionShape(b, hq, hkv, s, d)
        st.rotary = fa.RotaryEmbeddingConfig(THETA, 0) if kind == "gqa" else None
        if case.get("layout") == "projection":
            st.op = fa.HipProjectionRotaryGroupedPipeline(ctx, dtype)
        else:
            st.op = fa.HipRotaryGroupedAttention(ctx, dtype)
        st.bufs = [_buffer(t) for t in tensors]
        _output(st, st.op.layout(st.shape), tensors[0].shape, (b, hq, s), case["dtype"])
        if case.get("layout") == "prepared":
            torch.cuda.synchronize()
            ctx.set_prefill_precision(1 if case["precise"] else 0)
            st.prepared = st.op.prepare(*st.bufs, st.out, st.shape, st.config, st.rotary)
            ctx.set_prefill_precision(0)
        if kind == "train":
            st.backward = fa.HipGroupedBackwardRecomputePipeline(ctx, dtype)
            st.grads = [torch.empty_like(t) for t in tensors[:3]]
            st.grad_bufs = [_buffer(t) for t in st.grads]
    elif kind == "variable":
        n, hq, hkv, d = (case[x] for x in ("seqs", "q_heads", "kv_heads", "dim"))
        st.shape = fa.AsymmetricGroupedAttentionShape(n, hq, hkv, case["query"], case["kv"], d, 0)
        st.meta = [fa.VariableLengthSequenceMetadata(q, k, k - q, k - q) for q, k in _spans(case)]
        st.rotary = fa.VariableLengthRotaryEmbeddingConfig(THETA, 0)
        st.op = fa.HipVariableProjectionPipeline(ctx, dtype)
        st.bufs = [_buffer(t) for t in tensors]
        _output(st, st.op.layout(st.shape), tensors[0].shape, (n, hq, case["query"]),
                case["dtype"])
    elif kind == "resident":
        n, hq, hkv, d = (case[x] for x in ("batch", "q_heads", "kv_heads", "dim"))
        st.bufs = [_buffer(t) for t in tensors]
        st.plan = fa.ResidentDecodePlan(ctx, n, case["capacity"], case["live"], hq, hkv, d,
                                        st.config, THETA, case["live"] - 1, dtype)
        _output(st, st.plan.layout(), tensors[0].shape, (n, hq), case["dtype"])
    else:
        n, hq, hkv, d, page = (case[x] for x in ("seqs", "q_heads", "kv_heads", "dim", "page"))
        st.table, st.lens, st.total = tensors[-3:]
        st.bufs = [_buffer(t) for t in tensors[:-3]]
        if kind == "chunk":
            st.rotary = fa.RotaryEmbeddingConfig(THETA, 0)
            st.starts = np.full(n, case["cached"], np.int32)
            st.shape = fa.AsymmetricGroupedAttentionShape(
                n, hq, hkv, case["new"], case["cached"] + case["new"], d, case["cached"])
            st.plan = fa.PagedChunkedPrefillPlan(
                ctx, st.table, page, st.total, st.shape, st.config,
                fa.AsymmetricRotaryEmbeddingConfig(THETA, case["cached"], 0), dtype)
            _output(st, st.plan.layout(), tensors[0].shape, (n, hq, case["new"]), case["dtype"])
        elif kind == "decode":
            st.plan = fa.PagedDecodePlan(ctx, st.table, st.lens, page, st.total, hq, hkv, d,
                                         st.config, THETA, dtype)
            _output(st, st.plan.layout(), tensors[0].shape, (n, hq), case["dtype"])
        else:
            st.layout = fa.packed_layout(n * hq * d, n * hq, dtype)
            _output(st, st.layout, tensors[0].shape, (n, hq), case["dtype"])
    torch.cuda.synchronize()  # the inputs are made on torch's stream, the library has its own
    ctx.synchronize()
    return st


def run(st):
    case, kind = st.case, st.case["kind"]
    if kind == "mha":
        st.op.forward_resident(*st.bufs, st.shape, st.config, st.out)
    elif kind == "gqa":
        if case["layout"] == "prepared":
            st.op.encode_prepared(st.prepared)
        elif case["layout"] == "projection":
            st.op.encode(*st.bufs, st.out, st.shape, st.config, st.rotary)
        else:
            st.op.forward_resident(*st.bufs, st.shape, st.config, st.rotary, st.out)
    elif kind == "variable":
        st.op.encode(*st.bufs, st.out, st.shape, st.meta, st.config, st.rotary)
    elif kind in ("resident", "decode"):
        st.plan.launch(*st.bufs, st.out)
    elif kind == "step":
        fa.paged_decode_noalloc(_ctx(), st.table, st.lens, case["page"], st.total,
                                case["q_heads"], case["kv_heads"], case["dim"], st.config, THETA,
                                STORAGE[case["dtype"]], *st.bufs, st.out)
    elif kind == "chunk":
        q, k_pool, v_pool, k_new, v_new = st.bufs
        fa.paged_append_batched(_ctx(), st.table, st.starts, case["new"], case["page"], st.total,
                                case["kv_heads"], case["dim"], k_new, v_new, k_pool, v_pool,
                                st.rotary, STORAGE[case["dtype"]])
        st.plan.launch(q, k_pool, v_pool, st.out)
        return {"o": st.o, "lse": st.lse, "k": st.tensors[1], "v": st.tensors[2]}
    else:
        q, k, v, d_out = st.bufs
        st.op.forward_resident(q, k, v, st.shape, st.config, None, st.out)
        st.backward.encode_tensors(q, k, v, d_out, st.out, st.lse.data_ptr(), *st.grad_bufs,
                                   st.shape, st.config)
        return {"o": st.o, "lse": st.lse, "dq": st.grads[0], "dk": st.grads[1],
                "dv": st.grads[2]}
    return {"o": st.o, "lse": st.lse}


# ------------------------------------------------------------------------------- float64

def _rope(x, positions):
    """Interleaved RoPE of x [..., rows, dim] at `positions` [rows]. The frequencies and angles
    are f32 numbers by the operation's definition; the rest is float64."""
    d = x.shape[-1]
    theta, dim = np.float32(THETA), np.float32(d)
    freq = np.array([theta ** (np.float32(-2.0) * np.float32(j) / dim) for j in range(d // 2)],
                    np.float32)
    angle = positions.to(torch.float32).cpu().numpy()[:, None] * freq[None, :]
    angle = torch.from_numpy(angle.astype(np.float64)).to(x.device)
    cos, sin = torch.cos(angle), torch.sin(angle)
    even, odd = x[..., 0::2], x[..., 1::2]
    return torch.stack((even * cos - odd * sin, even * sin + odd * cos), -1).flatten(-2)


def _attend(q, k, v, first, d_out=None):
    """Attention of q [rows, d] over k, v [keys, d], row i seeing keys up to first + i (None: all).
    Returns O, LSE and, with d_out, (dQ, dK, dV)."""
    scale = 1.0 / math.sqrt(q.shape[-1])
    s = (q @ k.t().contiguous()) * scale
    if first is not None:
        rows = torch.arange(q.shape[0], device=q.device)[:, None] + first
        s.masked_fill_(torch.arange(k.shape[0], device=q.device)[None, :] > rows, -math.inf)
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse[:, None])
    o = p @ v
    if d_out is None:
        return o, lse, None
    ds = p * (d_out @ v.t().contiguous() - (d_out * o).sum(-1, keepdim=True))
    return o, lse, ((ds @ k) * scale, (ds.t().contiguous() @ q) * scale,
                    p.t().contiguous() @ d_out)


def exact(case, seed):
    tensors, _ = _inputs(case, seed)
    kind = case["kind"]
    dev = torch.device("cuda")
    if kind in ("mha", "gqa", "train"):
        q, k, v = (t.double() for t in tensors[:3])
        if case.get("layout") == "projection":
            q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
        b, hq, s, d = q.shape
        group = hq // k.shape[1]
        if kind == "gqa":
            positions = torch.arange(s)
            q, k = _rope(q, positions), _rope(k, positions)
        first = 0 if case["causal"] else None
        o, lse = torch.empty_like(q), torch.empty((b, hq, s), dtype=torch.float64, device=dev)
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for i in range(b):
            for h in range(hq):
                d_out = tensors[3][i, h].double() if kind == "train" else None
                o[i, h], lse[i, h], g = _attend(q[i, h], k[i, h // group], v[i, h // group],
                                                first, d_out)
                if g is not None:
                    dq[i, h] = g[0]
                    dk[i, h // group] += g[1]
                    dv[i, h // group] += g[2]
        if case.get("layout") == "projection":
            o = o.transpose(1, 2).contiguous()
        if kind == "train":
            return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
        return {"o": o, "lse": lse}

    q, k, v = (t.double() for t in tensors[:3])
    hq, hkv = case["q_heads"], case["kv_heads"]
    group = hq // hkv
    if kind == "variable":
        o = torch.zeros_like(q)
        lse = torch.full((case["seqs"], hq, case["query"]), -math.inf, dtype=torch.float64,
                         device=dev)
        for i, (nq, nk) in enumerate(_spans(case)):
            for h in range(hq):
                kk = _rope(k[i, :nk, h // group], torch.arange(nk))
                o[i, :nq, h], lse[i, h, :nq], _ = _attend(
                    _rope(q[i, :nq, h], torch.arange(nk - nq, nk)), kk, v[i, :nk, h // group],
                    nk - nq)
        return {"o": o, "lse": lse}

    if kind == "resident":
        n = case["batch"]
        keys = [(k[i, :case["live"]], v[i, :case["live"]]) for i in range(n)]
        lens = [case["live"]] * n
    else:
        table, lens, _total = tensors[-3:]
        n, page = case["seqs"], case["page"]
        if kind == "chunk":
            new = torch.arange(case["cached"], case["cached"] + case["new"])
            k_new, v_new = tensors[3].double(), tensors[4].double()
            at = table[:, new.numpy() // page]
            for i in range(n):
                rows = torch.from_numpy(at[i].astype(np.int64)).to(dev)
                offs = (new % page).to(dev)
                k[rows, offs] = _rope(k_new[i].transpose(0, 1), new).transpose(0, 1)
                v[rows, offs] = v_new[i]
        keys = []
        for i in range(n):
            pages = torch.from_numpy(table[i, :-(-int(lens[i]) // page)].astype(np.int64)).to(dev)
            keys.append(tuple(x[pages].reshape(-1, *x.shape[2:])[:int(lens[i])] for x in (k, v)))
    rows = case["new"] if kind == "chunk" else 1
    o = torch.empty((n, rows, hq, case["dim"]), dtype=torch.float64, device=dev)
    lse = torch.empty((n, hq, rows), dtype=torch.float64, device=dev)
    for i in range(n):
        length = int(lens[i])
        qi = _rope(q[i].view(rows, hq, -1).transpose(0, 1), torch.arange(length - rows, length))
        for h in range(hq):
            o[i, :, h], lse[i, h], _ = _attend(qi[h], keys[i][0][:, h // group].contiguous(),
                                               keys[i][1][:, h // group].contiguous(),
                                               length - rows)
    if kind == "chunk":
        return {"o": o, "lse": lse, "k": k, "v": v}
    return {"o": o.view(n, hq, -1), "lse": lse.view(n, hq)}


# ------------------------------------------------------------------------------- work, tolerance

def work(case):
    """Every input read once, every output written once; two operations per multiply-add over the
    visible (query, key) pairs, forward two products, backward five."""
    kind, d = case["kind"], case["dim"]
    size = TORCH[case["dtype"]].itemsize
    hq = case.get("q_heads", case.get("heads"))
    hkv = case.get("kv_heads", hq)
    if kind in ("mha", "gqa", "train"):
        b, s = case["batch"], case["seq"]
        pairs = b * (s * (s + 1) // 2 if case["causal"] else s * s)
        rows, keys = b * s, b * s
    elif kind == "variable":
        spans = _spans(case)
        pairs = sum(q * (k - q) + q * (q + 1) // 2 for q, k in spans)
        rows, keys = case["seqs"] * case["query"], sum(k for _, k in spans)
    elif kind == "chunk":
        n, new = case["seqs"], case["new"]
        pairs = n * (new * case["cached"] + new * (new + 1) // 2)
        rows, keys = n * new, n * (case["cached"] + new)
    else:
        lens = [case["live"]] * case["batch"] if kind == "resident" else _lengths(case).tolist()
        pairs = keys = sum(lens)
        rows = len(lens)
    nbytes = rows * hq * (2 * d * size + 4) + 2 * keys * hkv * d * size
    flops = 4 * pairs * hq * d
    if kind == "chunk":  # the new rows are written into the pools as well as read
        nbytes += 2 * rows * hkv * d * size
    if kind == "train":  # dO in, dQ, dK, dV out
        nbytes += rows * hq * 2 * d * size + 2 * keys * hkv * d * size
        flops += 10 * pairs * hq * d
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Relative error (2-norm) that another correct implementation at the same precision shows:
    about four times the largest that this library shows against float64 on the same inputs
    (bf16 3.4e-3, in O; f16 3.6e-4, in O; f32 9e-7, in dK)."""
    return {"rel": {"bf16": 1.2e-2, "f16": 1.5e-3, "f32": 4e-6}[case["dtype"]]}
