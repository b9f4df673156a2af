"""Performance cases: the work a program that uses this library has it do.

Seven kinds of call, each through the public entry points (``fellm_amd.ops``,
``fellm_amd.graph`` and the C functions of include/fellm_rocm.h):

  chain     prefill of one layer's memory-bound ops: embedding gather (dense or
            quantized table, alone or fused with RMSNorm), residual add +
            RMSNorm, RoPE of q and k, SwiGLU
  step      one continuous-batching decode step in one launch: RoPE + paged K/V
            append, residual add + RMSNorm, SwiGLU
  ffn       one token's feed-forward block on K-quant weights: gate/up GEMV +
            SwiGLU, then the down GEMV
  layer     one token's whole decode layer on K-quant weights, replayed from a
            HIP graph
  attn      paged decode attention of a batch of sequences of mixed lengths
  attn_f32  attention over contiguous f32 K/V: prefill rows, a canvas after a
            prefix, or one decode row
  moe       routing of a token batch: router, dispatch, gather, the experts'
            SwiGLU, weighted combine
"""
import math

import torch

import fellm_amd
from fellm_amd import graph, ops
from fellm_amd.abi import DeviceStepParams

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
# bytes and elements of one block of a quantized row
BLOCK = {"q4k": (144, 256), "q5k": (176, 256), "q6k": (210, 256), "q8_0": (34, 32)}


def listed():
    return [
        # A short f32 prompt at Llama-3.2-1B shape: four small launches from the host.
        {"name": "chain_1b_f32_t64", "kind": "chain", "tokens": 64, "hidden": 2048, "inter": 8192, "heads": 32,
         "kv_heads": 8, "head_dim": 64, "vocab": 128256, "act": "f32", "table": "dense", "fused": False, "pairing": 0},
        # Llama-3-8B prefill of 4096 tokens in f16.
        {"name": "chain_8b_f16_t4096", "kind": "chain", "tokens": 4096, "hidden": 4096, "inter": 14336, "heads": 32,
         "kv_heads": 8, "head_dim": 128, "vocab": 128256, "act": "f16", "table": "dense", "fused": False, "pairing": 0},
        # Qwen2-7B prefill from a Q6_K embedding table, a ragged token count, split-half RoPE, bf16.
        {"name": "chain_7b_q6k_t8191", "kind": "chain", "tokens": 8191, "hidden": 3584, "inter": 18944, "heads": 28,
         "kv_heads": 4, "head_dim": 128, "vocab": 152064, "act": "bf16", "table": "q6k", "fused": True, "pairing": 1},
        # Llama-3-70B serving step, 256 sequences, bf16 cache.
        {"name": "step_70b_bf16_b256", "kind": "step", "batch": 256, "hidden": 8192, "inter": 28672, "heads": 64,
         "kv_heads": 8, "head_dim": 128, "act": "bf16", "max_pos": 32768},
        # One token's feed-forward at Llama-3-70B shape, Q4_K with a Q6_K down projection.
        {"name": "ffn_70b_q4k_q6k", "kind": "ffn", "hidden": 8192, "inter": 28672, "up": "q4k", "down": "q6k"},
        # One token's decode layer at Llama-3-8B shape, Q4_K, 2048 keys: ten dependent launches.
        {"name": "layer_8b_q4k_s2048", "kind": "layer", "hidden": 4096, "inter": 14336, "heads": 32, "kv_heads": 8,
         "head_dim": 128, "seq": 2048, "weights": "q4k"},
        # One long sequence, Llama-3-8B heads, f16 cache.
        {"name": "attn_8b_b1_s32768", "kind": "attn", "batch": 1, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "max_seq": 32768, "act": "f16", "kv": "f16", "window": 0},
        # A serving batch of 256 sequences of up to 4096 keys, Llama-3-70B heads, bf16 cache.
        {"name": "attn_70b_b256_s4096", "kind": "attn", "batch": 256, "heads": 64, "kv_heads": 8, "head_dim": 128,
         "max_seq": 4096, "act": "bf16", "kv": "bf16", "window": 0},
        # Prefill of 512 rows against 2048 contiguous f32 keys, Llama-3-8B heads.
        {"name": "attn_f32_rows512", "kind": "attn_f32", "mode": "rows", "rows": 512, "keys": 2048, "heads": 32,
         "kv_heads": 8, "head_dim": 128},
        # One decode row against 4096 contiguous f32 keys.
        {"name": "attn_f32_decode_s4096", "kind": "attn_f32", "mode": "decode", "rows": 1, "keys": 4096, "heads": 32,
         "kv_heads": 8, "head_dim": 128},
        # Qwen3-30B-A3B MoE layer, 16384 tokens.
        {"name": "moe_30b_t16384", "kind": "moe", "tokens": 16384, "experts": 128, "top_k": 8, "hidden": 2048,
         "inter": 768},
        # The same layer for a decode batch of 64 tokens: launch latency.
        {"name": "moe_30b_t64", "kind": "moe", "tokens": 64, "experts": 128, "top_k": 8, "hidden": 2048, "inter": 768},
    ]


# ------------------------------------------------------------------------------ draws
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw(rng):
    kind = rng.choice(["chain", "step", "ffn", "layer", "attn", "attn", "attn_f32", "moe"])
    heads, kv_heads, head_dim = rng.choice([(32, 8, 64), (32, 8, 128), (28, 4, 128), (64, 8, 128), (32, 4, 128),
                                            (16, 4, 256), (16, 16, 64)])
    hidden = rng.choice([2048, 3072, 3584, 4096, 5120, 8192])
    if kind == "chain":
        table = rng.choice(["dense", "dense", "q4k", "q5k", "q6k", "q8_0"])
        return {"kind": kind, "tokens": _log(rng, 1, 8192), "hidden": hidden, "inter": 256 * rng.randint(16, 80),
                "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "vocab": rng.choice([32000, 128256]),
                "act": rng.choice(["f32", "f16", "bf16"]), "table": table, "fused": rng.random() < 0.5,
                "pairing": rng.choice([0, 1])}
    if kind == "step":
        return {"kind": kind, "batch": _log(rng, 1, 256), "hidden": hidden, "inter": 256 * rng.randint(16, 112),
                "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "act": rng.choice(["f16", "bf16"]),
                "max_pos": 4096}
    if kind == "ffn":
        return {"kind": kind, "hidden": hidden, "inter": 256 * rng.randint(20, 112),
                "up": rng.choice(["q4k", "q5k", "q6k"]), "down": rng.choice(["q4k", "q5k", "q6k"])}
    if kind == "layer":
        return {"kind": kind, "hidden": heads * head_dim, "inter": 256 * rng.randint(20, 64), "heads": heads,
                "kv_heads": kv_heads, "head_dim": head_dim, "seq": _log(rng, 16, 4096),
                "weights": rng.choice(["q4k", "q5k", "q6k"])}
    if kind == "attn":
        kv = rng.choice(["f16", "f16", "bf16"])
        return {"kind": kind, "batch": _log(rng, 1, 256), "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
                "max_seq": _log(rng, 64, 32768), "act": rng.choice([kv, "f32"]), "kv": kv,
                "window": rng.choice([0, 0, 0, 1024])}
    if kind == "attn_f32":
        mode = rng.choice(["rows", "canvas", "decode"])
        rows = 1 if mode == "decode" else _log(rng, 16, 512)
        return {"kind": kind, "mode": mode, "rows": rows, "keys": _log(rng, max(64, rows), 4096), "heads": heads,
                "kv_heads": kv_heads, "head_dim": head_dim}
    experts = rng.choice([8, 64, 128, 256])
    return {"kind": kind, "tokens": _log(rng, 1, 16384), "experts": experts,
            "top_k": rng.choice([2, 4, 8]) if experts > 8 else 2, "hidden": rng.choice([1024, 2048, 2880, 4096]),
            "inter": 64 * rng.randint(6, 24)}


def draw(rng):
    cap = max(work(c)["bytes"] for c in listed())
    while True:
        c = _draw(rng)
        w = work(c)
        if w["bytes"] <= cap and w["flops"] <= 40e9:
            return c


# ----------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    out = torch.empty(shape, dtype=dtype, device="cuda")
    return out.normal_(0.0, std, generator=g)


def _quant_table(g, qtype, rows, cols):
    """uint8 GGUF rows whose weights have a standard deviation near 0.02 and, for Q4_K / Q5_K, mean 0."""
    nbytes, nelem = BLOCK[qtype]
    nb = cols // nelem
    t = torch.randint(0, 256, (rows, nb, nbytes), generator=g, dtype=torch.uint8, device="cuda")
    u = 0.5 + torch.rand(rows, nb, generator=g, device="cuda")

    def put(at, v):
        t[..., at:at + 2] = v.to(torch.float16).view(torch.uint8).view(rows, nb, 2)

    if qtype in ("q4k", "q5k"):
        mid = 7.5 if qtype == "q4k" else 15.5
        d = u * (1e-3 / mid)
        put(0, d)
        put(2, d * mid)
    elif qtype == "q6k":
        sc = torch.randint(-32, 33, (rows, nb, 16), generator=g, dtype=torch.int8, device="cuda")
        t[..., 192:208] = sc.view(torch.uint8)
        put(208, u * 6e-5)
    else:
        put(0, u * 2.7e-4)
    return t.view(rows, nb * nbytes)


def _zipf(g, n, vocab, s=1.1):
    cdf = torch.cumsum(torch.arange(1, vocab + 1, dtype=torch.float64, device="cuda") ** -s, 0)
    u = torch.rand(n, generator=g, dtype=torch.float64, device="cuda") * cdf[-1]
    return torch.searchsorted(cdf, u).clamp_(max=vocab - 1).to(torch.int32)


def _norm_weight(g, n):
    return 1.0 + 0.1 * _randn(g, n)


def _inv_freqs(head_dim):
    return ops.rope_inv_freqs(500000.0, head_dim).cuda()


def _paged_cache(g, lens, kv_heads, head_dim, kv, fill=True):
    """A cache that holds lens[b] tokens of row b, physical blocks in random order."""
    stride = kv_heads * head_dim
    block_bytes = ops.PagedKvCache.block_bytes_for(stride)
    n_logical = max((max(lens) + 15) // 16, 1)
    need = [(n + 15) // 16 for n in lens]
    blocks = max(sum(need), 1)
    arena = torch.zeros(blocks * block_bytes, dtype=torch.uint8, device="cuda")
    if fill:
        arena.view(DT[kv]).normal_(0.0, 0.5, generator=g)
    order = torch.randperm(blocks, generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(len(lens), n_logical, dtype=torch.int32, device="cuda")
    need_t = torch.tensor(need, device="cuda")
    used = torch.arange(n_logical, device="cuda")[None, :] < need_t[:, None]
    table[used] = order[:sum(need)]
    return ops.PagedKvCache(arena=arena, block_table=table.view(-1), n_layers=1, n_logical_blocks=n_logical,
                            block_size=16, block_bytes=block_bytes, stride=stride, kv_dtype=DT[kv])


def _lengths(c, seed):
    """Sequence lengths of a serving batch: uniform over the longest sixteenth's multiples, one of them the longest."""
    g = torch.Generator()
    g.manual_seed(seed + 77)
    lo = max(c["max_seq"] // 16, 1)
    lens = torch.randint(lo, c["max_seq"] + 1, (c["batch"],), generator=g).tolist()
    lens[0] = c["max_seq"]
    return lens


def _inputs(c, seed):
    g = _gen(seed)
    k = c["kind"]
    s = {"c": c}
    if k == "chain":
        T, H, dt = c["tokens"], c["hidden"], DT[c["act"]]
        qw, kw = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        if c["table"] == "dense":
            s["table"] = _randn(g, c["vocab"], H, std=0.02, dtype=dt)
            s["ids"] = torch.randint(0, c["vocab"], (T,), generator=g, device="cuda", dtype=torch.int32)
        else:
            s["table"] = _quant_table(g, c["table"], c["vocab"], H)
            s["ids"] = _zipf(g, T, c["vocab"])
        s["w0"], s["w1"], s["inv"] = _norm_weight(g, H), _norm_weight(g, H), _inv_freqs(c["head_dim"])
        s["pos"] = torch.arange(T, dtype=torch.int32, device="cuda")
        s["x"], s["q"], s["k"] = (_randn(g, T, n, dtype=dt) for n in (H, qw, kw))
        s["gate"], s["up"] = (_randn(g, T, c["inter"], dtype=dt) for _ in range(2))
    elif k == "step":
        B, H, dt = c["batch"], c["hidden"], DT[c["act"]]
        qw, kw = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        s["pos"] = torch.randint(0, c["max_pos"], (B,), generator=g, device="cuda", dtype=torch.int32)
        # each row's current block is its own; the other entries are never touched by an append
        n_logical, bb = (c["max_pos"] + 15) // 16, ops.PagedKvCache.block_bytes_for(kw)
        table = torch.zeros(B, n_logical, dtype=torch.int32, device="cuda")
        table[torch.arange(B, device="cuda"), s["pos"].long() // 16] = torch.randperm(
            B, generator=g, device="cuda").to(torch.int32)
        s["cache"] = ops.PagedKvCache(arena=torch.zeros(B * bb, dtype=torch.uint8, device="cuda"),
                                      block_table=table.view(-1), n_layers=1, n_logical_blocks=n_logical,
                                      block_size=16, block_bytes=bb, stride=kw, kv_dtype=dt)
        s["w0"], s["inv"] = _norm_weight(g, H), _inv_freqs(c["head_dim"])
        s["q"], s["k"], s["v"], s["x"] = (_randn(g, B, n, dtype=dt) for n in (qw, kw, kw, H))
        s["r"] = _randn(g, B, H, std=2.0, dtype=dt)
        s["gate"], s["up"] = (_randn(g, B, c["inter"], dtype=dt) for _ in range(2))
    elif k == "ffn":
        H, I = c["hidden"], c["inter"]
        s["g"], s["u"] = (_quant_table(g, c["up"], I, H) for _ in range(2))
        s["d"] = _quant_table(g, c["down"], H, I)
        s["x"] = _randn(g, H)
    elif k == "layer":
        H, I, kw = c["hidden"], c["inter"], c["kv_heads"] * c["head_dim"]
        for name, rows, cols in (("qkv", H + 2 * kw, H), ("o", H, H), ("g", I, H), ("u", I, H), ("d", H, I)):
            s["w_" + name] = _quant_table(g, c["weights"], rows, cols)
        s["n1"], s["n2"], s["inv"] = _norm_weight(g, H), _norm_weight(g, H), _inv_freqs(c["head_dim"])
        s["cache"] = _paged_cache(g, [c["seq"]], c["kv_heads"], c["head_dim"], "f16")
        s["x"] = _randn(g, 1, H)
    elif k == "attn":
        s["lens"] = _lengths(c, seed)
        s["cache"] = _paged_cache(g, s["lens"], c["kv_heads"], c["head_dim"], c["kv"])
        s["q"] = _randn(g, c["batch"], c["heads"] * c["head_dim"], dtype=DT[c["act"]])
        s["len_dev"] = torch.tensor(s["lens"], dtype=torch.int32, device="cuda")
    elif k == "attn_f32":
        kw = c["kv_heads"] * c["head_dim"]
        # rows mode reads q head-major, the others row-major: the same count of values
        s["q"] = _randn(g, c["rows"] * c["heads"] * c["head_dim"])
        s["k"], s["v"] = _randn(g, c["keys"], kw), _randn(g, c["keys"], kw)
        if c["mode"] == "canvas":
            s["k2"], s["v2"] = _randn(g, c["rows"], kw), _randn(g, c["rows"], kw)
    else:
        T, E, K, H = c["tokens"], c["experts"], c["top_k"], c["hidden"]
        s["logits"] = _randn(g, T, E) + _randn(g, 1, E, std=0.5)
        s["x"] = _randn(g, T, H, dtype=torch.bfloat16)
        s["gate"], s["up"] = (_randn(g, T * K, c["inter"], dtype=torch.bfloat16) for _ in range(2))
        s["eo"], s["y0"] = _randn(g, T * K, H), _randn(g, T, H)
    return s


def prepare(case, seed):
    c = dict(case)
    s = _inputs(c, seed)
    if c["kind"] == "chain":
        s["emb"] = torch.empty_like(s["x"])
        s["outs"] = {n: torch.empty_like(s[n if n in s else "x"]) for n in ("h", "y", "y0", "q", "k")}
        s["outs"]["act"] = torch.empty_like(s["gate"])
    elif c["kind"] == "step":
        s["outs"] = {"q_out": torch.empty_like(s["q"]), "h_out": torch.empty_like(s["x"]),
                     "y_out": torch.empty_like(s["x"]), "act_out": torch.empty_like(s["gate"])}
    elif c["kind"] == "attn_f32":
        s["out"] = torch.empty_like(s["q"])
    elif c["kind"] == "layer":
        _capture_layer(c, s)
    return s


def _capture_layer(c, s):
    H, hd, nh, nkv = c["hidden"], c["head_dim"], c["heads"], c["kv_heads"]
    kw = nkv * hd
    max_seq = s["cache"].n_logical_blocks * 16
    params = DeviceStepParams(token_id=0, position=c["seq"] - 1, sequence_length=c["seq"], active_batch=1,
                              kv_write_slot=(c["seq"] - 1) % 16)
    s["params"] = torch.frombuffer(bytearray(bytes(params)), dtype=torch.uint8).cuda()
    ws = fellm_amd.lib().fellm_rocm_paged_attention_workspace(1, nh, nkv, hd, max_seq)
    f = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    b = {"y": f(1, H), "qkv": f(H + 2 * kw), "q": f(1, H), "att": f(1, H), "o": f(H), "h": f(1, H), "y2": f(1, H),
         "act": f(c["inter"]), "down": f(H), "out": f(1, H), "ws": f(max(ws // 4, 1)),
         "pos": torch.empty(1, dtype=torch.int32, device="cuda")}
    s["b"] = b
    qt, qkv = c["weights"], b["qkv"]
    q, k, v = qkv[:H].view(1, H), qkv[H:H + kw].view(1, kw), qkv[H + kw:].view(1, kw)

    def layer():
        ops.rmsnorm(s["x"], s["n1"], 1e-5, out=b["y"])
        ops.matvec_kquant(s["w_qkv"], b["y"].view(-1), qtype=qt, out=qkv)
        ops.step_kv_position(s["params"], 16, out=b["pos"])
        ops.rope_kv_write(q, k, v, s["inv"], b["pos"], s["cache"], head_dim=hd,
                          rope_positions=ops.step_field(s["params"], "position"), q_out=b["q"])
        ops.paged_attention(b["q"], ops.step_field(s["params"], "sequence_length"), s["cache"], n_heads=nh,
                            n_kv_heads=nkv, head_dim=hd, max_seq=max_seq, out=b["att"], workspace=b["ws"])
        ops.matvec_kquant(s["w_o"], b["att"].view(-1), qtype=qt, out=b["o"])
        ops.add_rmsnorm(b["o"].view(1, H), s["x"], s["n2"], 1e-5, h_out=b["h"], y_out=b["y2"])
        ops.gate_up_swiglu(s["w_g"], s["w_u"], b["y2"].view(-1), qtype=qt, out=b["act"])
        ops.matvec_kquant(s["w_d"], b["act"].view(-1), qtype=qt, out=b["down"])
        ops.add(b["down"].view(1, H), b["h"], out=b["out"])

    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream), graph.GraphCapture(stream) as cap:
        layer()
    s["graph"] = cap.graph


# ------------------------------------------------------------------------------- runs
def run(s):
    c = s["c"]
    return _RUN[c["kind"]](c, s)


def _run_chain(c, s):
    o = s["outs"]
    kw = {"dim": c["hidden"], "qtype": None if c["table"] == "dense" else c["table"]}
    if c["fused"]:
        ops.embedding_rmsnorm(s["table"], s["ids"], s["w0"], 1e-6, h_out=s["emb"], y_out=o["y0"], **kw)
    else:
        ops.embedding(s["table"], s["ids"], out=s["emb"], **kw)
    ops.add_rmsnorm(s["x"], s["emb"], s["w1"], 1e-5, h_out=o["h"], y_out=o["y"])
    ops.rope(s["q"], s["inv"], head_dim=c["head_dim"], pairing=c["pairing"], positions=s["pos"], x2=s["k"],
             out1=o["q"], out2=o["k"])
    ops.silu_gate(s["gate"], s["up"], out=o["act"])
    r = [s["emb"], o["h"], o["y"], o["q"], o["k"], o["act"]]
    return r + [o["y0"]] if c["fused"] else r


def _run_step(c, s):
    out = ops.decode_step(s["q"], s["k"], s["v"], s["inv"], s["pos"], s["cache"], s["x"], s["r"], s["w0"], 1e-5,
                          s["gate"], s["up"], head_dim=c["head_dim"], **s["outs"])
    return [*out, s["cache"].arena.view(DT[c["act"]])]


def _run_ffn(c, s):
    act = ops.gate_up_swiglu(s["g"], s["u"], s["x"], qtype=c["up"])
    return [act, ops.matvec_kquant(s["d"], act, qtype=c["down"])]


def _run_layer(c, s):
    s["graph"].launch()
    b = s["b"]
    return [b["q"], b["att"], b["h"], b["act"], b["out"]]


def _run_attn(c, s):
    return ops.paged_attention(s["q"], s["len_dev"], s["cache"], n_heads=c["heads"], n_kv_heads=c["kv_heads"],
                               head_dim=c["head_dim"], max_seq=c["max_seq"], window=c["window"])


def _run_attn_f32(c, s):
    lib, stream = fellm_amd.lib(), torch.cuda.current_stream().cuda_stream
    q, out, k, v = (s[n].data_ptr() for n in ("q", "out", "k", "v"))
    nh, nkv, hd = c["heads"], c["kv_heads"], c["head_dim"]
    if c["mode"] == "rows":
        rc = lib.fellm_rocm_attention_f32kv_rows(q, out, c["rows"], nh, nkv, hd, k, v, c["keys"], 0.0, 1, 0, stream)
    else:
        k2, v2 = (s[n].data_ptr() if n in s else None for n in ("k2", "v2"))
        rc = lib.fellm_rocm_attention_f32kv(q, out, c["rows"], nh, nkv, hd, k, v, 0, c["keys"], k2, v2,
                                            c["rows"] if k2 else 0, 0.0, stream)
    if rc:
        raise RuntimeError("attention_f32kv: %d" % rc)
    return s["out"]


def _run_moe(c, s):
    ids, weights = ops.router_topk(s["logits"], c["top_k"])
    d = ops.moe_dispatch(ids, c["experts"])
    grouped = ops.moe_gather(s["x"], d.order, c["top_k"], inv=d.inv)
    act = ops.silu_gate(s["gate"], s["up"])
    y = ops.moe_combine(s["eo"], weights, ids=ids, inv=d.inv, y0=s["y0"])
    return [ids, weights, d.counts, d.offsets, d.order, d.inv, grouped, act, y]


_RUN = {"chain": _run_chain, "step": _run_step, "ffn": _run_ffn, "layer": _run_layer, "attn": _run_attn,
        "attn_f32": _run_attn_f32, "moe": _run_moe}


# ------------------------------------------------------------------- work and tolerance
def _row_bytes(qtype, cols):
    nbytes, nelem = BLOCK[qtype]
    return cols // nelem * nbytes


def work(case):
    c, k = case, case["kind"]
    if k == "chain":
        T, H, e = c["tokens"], c["hidden"], SIZE[c["act"]]
        row = H * e if c["table"] == "dense" else _row_bytes(c["table"], H)
        heads = (c["heads"] + c["kv_heads"]) * c["head_dim"]
        rows = row + 4 + H * e * (2 if c["fused"] else 1) + 4 * H * e + 2 * heads * e + 4 + 3 * c["inter"] * e
        return {"bytes": T * rows, "flops": T * (6 * H + 3 * heads + 6 * c["inter"])}
    if k == "step":
        B, H, e = c["batch"], c["hidden"], SIZE[c["act"]]
        qw, kw = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        return {"bytes": B * e * (2 * qw + 4 * kw + 4 * H + 3 * c["inter"]),
                "flops": B * (3 * (qw + kw) + 4 * H + 6 * c["inter"])}
    if k == "ffn":
        H, I = c["hidden"], c["inter"]
        return {"bytes": 2 * I * _row_bytes(c["up"], H) + H * _row_bytes(c["down"], I) + 4 * (2 * H + 2 * I),
                "flops": 6 * H * I}
    if k == "layer":
        H, I, kw = c["hidden"], c["inter"], c["kv_heads"] * c["head_dim"]
        weights = (2 * H + 2 * kw + 2 * I) * _row_bytes(c["weights"], H) + H * _row_bytes(c["weights"], I)
        return {"bytes": weights + 4 * kw * c["seq"] + 4 * 8 * H,
                "flops": 2 * H * (2 * H + 2 * kw + 3 * I) + 4 * H * c["seq"]}
    if k == "attn":
        kw, qw = c["kv_heads"] * c["head_dim"], c["heads"] * c["head_dim"]
        lens = _lengths(c, 0)
        keys = sum(min(n, c["window"] or n) for n in lens)
        return {"bytes": keys * kw * 4 + 2 * c["batch"] * qw * SIZE[c["act"]], "flops": 4 * qw * keys}
    if k == "attn_f32":
        qw, kw, n, r = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["keys"], c["rows"]
        pairs = {"rows": r * n - r * (r - 1) // 2, "canvas": r * (n + r), "decode": n}[c["mode"]]
        keys = n + r if c["mode"] == "canvas" else n
        return {"bytes": 8 * (keys * kw + r * qw), "flops": 4 * qw * pairs}
    T, A, H = c["tokens"], c["tokens"] * c["top_k"], c["hidden"]
    by = T * c["experts"] * 4 + A * 8 + A * 12 + 8 * c["experts"]   # router, dispatch
    by += A * 8 + (T + A) * H * 2 + A * c["inter"] * 6              # gather, SwiGLU
    return {"bytes": by + A * 12 + (A + 2 * T) * H * 4, "flops": 2 * A * H + 6 * A * c["inter"]}


def tolerance(case):
    # 16-bit results: their rounding (2^-11, 2^-8 a value at most); f32 results: sums in another order.
    k = case["kind"]
    if k in ("chain", "step", "attn"):
        rel = {"f32": 1e-5, "f16": 1e-3, "bf16": 8e-3}
        return {"rel": rel[case["act"]], "max": 10 * rel[case["act"]]}
    if k == "moe":
        return {"rel": 8e-3, "max": 8e-2, "differ": 1e-4}
    if k == "ffn":
        # a different rounding moves an activation over a quantization step now and then
        return {"rel": 1e-3, "max": 5e-2}
    if k == "layer":
        return {"rel": 2e-3, "max": 5e-2}
    return {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------------- 64-bit results
def _dequant(t, qtype):
    """f64 values of uint8 GGUF rows."""
    nbytes, nelem = BLOCK[qtype]
    rows = t.shape[0]
    b = t.view(rows, -1, nbytes)
    nb = b.shape[1]

    def half(at):
        return b[..., at:at + 2].contiguous().view(torch.float16).double()

    if qtype == "q8_0":
        return (half(0) * b[..., 2:].contiguous().view(torch.int8).double()).view(rows, -1)
    if qtype == "q6k":
        ql, qh = b[..., :128].view(rows, nb, 2, 2, 32).int(), b[..., 128:192].view(rows, nb, 2, 1, 32).int()
        low = torch.stack([ql & 15, ql >> 4], 3).view(rows, nb, 2, 4, 32)
        high = (qh >> torch.tensor([0, 2, 4, 6], device=t.device).view(4, 1)) & 3
        q = (low + 16 * high - 32).view(rows, nb, 16, 16).double()
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        q *= (half(208) * sc).unsqueeze(-1)
        return q.view(rows, -1)
    s = b[..., 4:16].int()
    lo, mi, hi = s[..., :4], s[..., 4:8], s[..., 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1).double()
    mn = torch.cat([mi & 63, (hi >> 4) | ((mi >> 6) << 4)], -1).double()
    qs = b[..., -128:].view(rows, nb, 4, 1, 32).int()
    q = torch.cat([qs & 15, qs >> 4], 3).view(rows, nb, 8, 32)
    if qtype == "q5k":
        qh = b[..., 16:48].view(rows, nb, 1, 32).int()
        q = q + 16 * ((qh >> torch.arange(8, device=t.device).view(8, 1)) & 1)
    q = q.double()
    q *= (half(0) * sc).unsqueeze(-1)
    q -= (half(2) * mn).unsqueeze(-1)
    return q.view(rows, -1)


def _q8k(x):
    """x as its 8-bit blocks of 256 hold it."""
    b = x.double().view(-1, 256)
    amax = b.abs().amax(1, keepdim=True).clamp_min(1e-300)
    return (torch.round(b * (127.0 / amax)).clamp(-128, 127) * (amax / 127.0)).view(-1)


def _gemv(w, qtype, x):
    y, xq = [], _q8k(x)
    for part in w.split(4096):
        y.append(_dequant(part, qtype) @ xq)
    return torch.cat(y)


def _silu(g, u):
    g = g.double()
    return g / (1.0 + torch.exp(-g)) * u.double()


def _rms(h, w, eps):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, head_dim, inv, pos, pairing):
    rows = x.shape[0]
    theta = (pos.float()[:, None] * inv[None, :]).double()[:, None, :]
    s, c = torch.sin(theta), torch.cos(theta)
    v = x.double().view(rows, -1, head_dim)
    if pairing == 0:
        a, b = v[..., 0::2], v[..., 1::2]
        return torch.stack([a * c - b * s, a * s + b * c], -1).view(rows, -1)
    a, b = v[..., :head_dim // 2], v[..., head_dim // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1).view(rows, -1)


def _keys(cache, row, lo, n, which):
    """f64 rows lo .. n-1 of sequence `row`'s K (0) or V (1)."""
    st = cache.stride
    blocks = cache.block_table.view(-1, cache.n_logical_blocks)[row, :(n + 15) // 16].long()
    a = cache.arena.view(cache.kv_dtype).view(-1, cache.block_bytes // 2)[blocks]
    a = a[:, which * 16 * st:(which + 1) * 16 * st].reshape(-1, st)
    return a[lo:n].double()


def _attend(q, k, v, kv_heads, head_dim, mask=None):
    """q [rows, heads * head_dim] against k, v [keys, kv_heads * head_dim], all f64."""
    rows, n = q.shape[0], k.shape[0]
    heads = q.shape[1] // head_dim
    G = heads // kv_heads
    qh = q.view(rows, kv_heads, G, head_dim).permute(1, 2, 0, 3).reshape(kv_heads, G * rows, head_dim)
    kh = k.view(n, kv_heads, head_dim).permute(1, 2, 0).contiguous()
    vh = v.view(n, kv_heads, head_dim).permute(1, 0, 2).contiguous()
    sc = torch.matmul(qh, kh) * (1.0 / math.sqrt(head_dim))
    if mask is not None:
        sc = sc.view(kv_heads, G, rows, n).masked_fill(~mask, -math.inf).view(kv_heads, G * rows, n)
    o = torch.matmul(torch.softmax(sc, -1), vh)
    return o.view(kv_heads, G, rows, head_dim).permute(2, 0, 1, 3).reshape(rows, -1)


def exact(case, seed):
    c = dict(case)
    s = _inputs(c, seed)
    return _EXACT[c["kind"]](c, s)


def _exact_chain(c, s):
    rows = s["table"][s["ids"].long()]
    emb = rows.double() if c["table"] == "dense" else _dequant(rows, c["table"])
    h = s["x"].double() + emb
    r = [emb, h, _rms(h, s["w1"], 1e-5), _rope(s["q"], c["head_dim"], s["inv"], s["pos"], c["pairing"]),
         _rope(s["k"], c["head_dim"], s["inv"], s["pos"], c["pairing"]), _silu(s["gate"], s["up"])]
    return r + [_rms(emb, s["w0"], 1e-6)] if c["fused"] else r


def _exact_step(c, s):
    h = s["x"].double() + s["r"].double()
    cache, pos, kw = s["cache"], s["pos"].long(), c["kv_heads"] * c["head_dim"]
    arena = torch.zeros(cache.arena.numel() // cache.block_bytes, cache.block_bytes // 2, dtype=torch.float64,
                        device="cuda")
    k = _rope(s["k"], c["head_dim"], s["inv"], s["pos"], 0)
    blocks = cache.block_table.view(-1, cache.n_logical_blocks)[torch.arange(c["batch"], device="cuda"), pos // 16]
    at = torch.arange(kw, device="cuda")[None, :] + (pos % 16)[:, None] * kw
    arena[blocks.long()[:, None], at] = k
    arena[blocks.long()[:, None], at + 16 * kw] = s["v"].double()
    return [_rope(s["q"], c["head_dim"], s["inv"], s["pos"], 0), h, _rms(h, s["w0"], 1e-5),
            _silu(s["gate"], s["up"]), arena.view(-1)]


def _exact_ffn(c, s):
    act = _silu(_gemv(s["g"], c["up"], s["x"]), _gemv(s["u"], c["up"], s["x"]))
    return [act, _gemv(s["d"], c["down"], act)]


def _exact_layer(c, s):
    H, hd, kw, qt, n = c["hidden"], c["head_dim"], c["kv_heads"] * c["head_dim"], c["weights"], c["seq"]
    x = s["x"].double()
    qkv = _gemv(s["w_qkv"], qt, _rms(x, s["n1"], 1e-5).view(-1))
    pos = torch.tensor([n - 1], device="cuda")
    q, k = (_rope(t.view(1, -1), hd, s["inv"], pos, 0) for t in (qkv[:H], qkv[H:H + kw]))
    keys, vals = (_keys(s["cache"], 0, 0, n, w) for w in (0, 1))
    keys[n - 1], vals[n - 1] = k.half().double(), qkv[H + kw:].half().double()
    att = _attend(q, keys, vals, c["kv_heads"], hd)
    h = _gemv(s["w_o"], qt, att.view(-1)).view(1, H) + x
    y = _rms(h, s["n2"], 1e-5).view(-1)
    act = _silu(_gemv(s["w_g"], qt, y), _gemv(s["w_u"], qt, y))
    return [q, att, h, act, _gemv(s["w_d"], qt, act).view(1, H) + h]


def _exact_attn(c, s):
    out = []
    for row, n in enumerate(s["lens"]):
        lo = max(n - c["window"], 0) if c["window"] else 0
        k, v = (_keys(s["cache"], row, lo, n, w) for w in (0, 1))
        out.append(_attend(s["q"][row:row + 1].double(), k, v, c["kv_heads"], c["head_dim"]))
    return torch.cat(out)


def _exact_attn_f32(c, s):
    r, n, nh, hd = c["rows"], c["keys"], c["heads"], c["head_dim"]
    q, k, v, mask = s["q"].double(), s["k"].double(), s["v"].double(), None
    if c["mode"] == "rows":
        q = q.view(nh, r, hd).permute(1, 0, 2).reshape(r, nh * hd)
        at = torch.arange(n, device="cuda")[None, :] - torch.arange(r, device="cuda")[:, None]
        mask = at <= n - r
    elif c["mode"] == "canvas":
        k, v = torch.cat([k, s["k2"].double()]), torch.cat([v, s["v2"].double()])
    o = _attend(q.view(r, nh * hd), k, v, c["kv_heads"], hd, mask)
    return (o.view(r, nh, hd).permute(1, 0, 2) if c["mode"] == "rows" else o).reshape(-1)


def _exact_moe(c, s):
    T, K = c["tokens"], c["top_k"]
    p, ids = torch.softmax(s["logits"].double(), -1).topk(K, -1)
    order = torch.argsort(ids.reshape(-1), stable=True)
    inv = torch.empty_like(order)
    inv[order] = torch.arange(T * K, device="cuda")
    w = p / p.sum(-1, keepdim=True)
    y = s["y0"].double()
    for k in range(K):
        y += w[:, k:k + 1] * s["eo"][inv.view(T, K)[:, k]].double()
    return [None, w, None, None, None, None, s["x"][order // K].double(), _silu(s["gate"], s["up"]), y]


_EXACT = {"chain": _exact_chain, "step": _exact_step, "ffn": _exact_ffn, "layer": _exact_layer, "attn": _exact_attn,
          "attn_f32": _exact_attn_f32, "moe": _exact_moe}
