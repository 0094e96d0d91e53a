"""The work a user of this library has it do, as measurable cases.

Every case goes through the public entry points: the attention layer with the forward context the engine
sets, the int8 linears, the norm / RoPE / activation layers, the draft model and the rejection-sampling
verification. Geometries are the library's own: attention with 32 or 16 query heads over 8 kv heads of 128,
256-token pages, decoder layers of hidden 1024 / intermediate 3072 and 2560 / 9728, vocabulary 151936.
Work of a few rows (decode) runs from a captured HIP graph, as the engine replays it; prefills,
attention over a batch and the verification run eagerly.
"""
from __future__ import annotations

import math

import torch

import __graft_entry__

__graft_entry__.load_package()

from specdec_nanovllm_amd import ops  # noqa: E402
from specdec_nanovllm_amd.draft_chain import DraftChain  # noqa: E402
from specdec_nanovllm_amd.layers.activation import SiluAndMul  # noqa: E402
from specdec_nanovllm_amd.layers.attention import Attention  # noqa: E402
from specdec_nanovllm_amd.layers.layernorm import RMSNorm  # noqa: E402
from specdec_nanovllm_amd.layers.linear import ReplicatedLinear  # noqa: E402
from specdec_nanovllm_amd.spec_decode.verify import verify_batch  # noqa: E402
from specdec_nanovllm_amd.utils.context import set_context  # noqa: E402

D = 128          # head_dim
KV_HEADS = 8
PAGE = 256
VOCAB = 151936
EPS = 1e-6
GROUP = 128      # columns per scale of the per-group format
LAYERS = 28      # the draft model's
SMALL = dict(hidden=1024, inter=3072, heads=16)
LARGE = dict(hidden=2560, inter=9728, heads=32)
GRAPH_ROWS = 64  # linears of up to this many rows are decode work: replayed from a graph
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


# ------------------------------------------------------------------------------------- cases
def listed():
    return [
        # one user's draft model proposing a token: the latency of speculative decoding
        dict(name="draft_step_b1", kind="draft", batch=1, ctx=2048),
        # the same for a batch of users
        dict(name="draft_step_b16", kind="draft", batch=16, ctx=2048),
        # one attention layer of the target model's decode step, contexts of all lengths
        dict(name="decode_b32", kind="decode", batch=32, lo=512, hi=4096, heads=32, dtype="bf16"),
        # few users with long contexts
        dict(name="decode_long_b3", kind="decode", batch=3, lo=8192, hi=32768, heads=32, dtype="bf16"),
        # one attention layer of the target model verifying 6 drafted tokens per sequence
        dict(name="verify_b8", kind="verify", batch=8, k=6, lo=1500, hi=2600, heads=32, dtype="bf16"),
        # one attention layer prefilling four prompts
        dict(name="prefill_4x2048", kind="prefill", batch=4, lo=2048, hi=2048, cached=0, heads=32, dtype="bf16"),
        # prompts of odd lengths whose beginnings are already in the pages (prefix cache)
        dict(name="prefill_cached_b5", kind="prefill", batch=5, lo=130, hi=1700, cached=1024, heads=16, dtype="fp16"),
        # a whole int8 decoder layer of the draft model over prompts of odd lengths
        dict(name="layer_prefill_b5", kind="layer", batch=5, lo=300, hi=2000, dtype="bf16"),
        # the target model's int8 MLP over a full prefill batch
        dict(name="mlp_4096", kind="mlp", rows=4096, size="large", group=0, dtype="bf16"),
        # the same MLP for the 56 rows of a verify step (8 sequences x 7)
        dict(name="mlp_56", kind="mlp", rows=56, size="large", group=0, dtype="bf16"),
        # final norm and vocabulary projection of a verify step
        dict(name="head_56", kind="head", rows=56, dtype="bf16"),
        # accepting or rejecting 6 drafted tokens for 8 sequences
        dict(name="accept_b8", kind="accept", batch=8, k=6, dtype="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["draft", "decode", "decode", "verify", "prefill", "prefill", "layer", "mlp", "mlp", "mlp",
                       "head", "accept"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    heads = rng.choice([16, 32])
    if kind == "draft":
        return dict(kind=kind, batch=_log_int(rng, 1, 16), ctx=_log_int(rng, 100, 2048))
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        hi = _log_int(rng, 100, min(32768, 131072 // batch))
        return dict(kind=kind, batch=batch, lo=max(1, int(hi * rng.uniform(0.1, 1.0))), hi=hi, heads=heads, dtype=dtype)
    if kind == "verify":
        hi = _log_int(rng, 200, 4096)
        return dict(kind=kind, batch=_log_int(rng, 1, 16), k=rng.randint(2, 7), lo=max(20, int(hi * rng.uniform(0.2, 1.0))),
                    hi=hi, heads=heads, dtype=dtype)
    if kind == "prefill":
        batch = _log_int(rng, 1, 8)
        hi = _log_int(rng, 40, 8192 // batch)
        return dict(kind=kind, batch=batch, lo=max(1, int(hi * rng.uniform(0.2, 1.0))), hi=hi,
                    cached=rng.choice([0, 0, PAGE * rng.randint(1, 8)]), heads=heads, dtype=dtype)
    if kind == "layer":
        batch = _log_int(rng, 1, 8)
        hi = _log_int(rng, 40, 8192 // batch)
        return dict(kind=kind, batch=batch, lo=max(1, int(hi * rng.uniform(0.2, 1.0))), hi=hi, dtype=dtype)
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 1, 4096), size=rng.choice(["small", "large"]),
                    group=rng.choice([0, 0, GROUP]), dtype=dtype)
    if kind == "head":
        return dict(kind=kind, rows=_log_int(rng, 1, 128), dtype=dtype)
    return dict(kind=kind, batch=_log_int(rng, 1, 16), k=rng.randint(2, 7), dtype=rng.choice(["fp32", "bf16"]))


# ------------------------------------------------------------------------------------ inputs
def _gens(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g, torch.Generator().manual_seed(seed + 1)


def _randn(g, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _lens(case, cg):
    """Lengths in [lo, hi], the longest among them (as the case's own numbers give them)."""
    n = torch.randint(case["lo"], case["hi"] + 1, (case["batch"],), generator=cg)
    n[int(torch.randint(0, case["batch"], (1,), generator=cg))] = case["hi"]
    return n.tolist()


def _case_lens(case):
    """The lengths that work() counts: the sizes of a case are the same for every seed."""
    return _lens(case, torch.Generator().manual_seed(1234 + case["batch"]))


def _pages(g, cg, keys, dtype):
    """Paged caches holding ``keys`` tokens per sequence on shuffled pages, and the block table."""
    need = [-(-n // PAGE) for n in keys]
    perm = torch.randperm(sum(need) + 2, generator=cg).to(torch.int32)
    bt = torch.full((len(keys), max(need)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n]
        at += n
    shape = (sum(need) + 2, PAGE, KV_HEADS, D)
    return _randn(g, shape, dtype), _randn(g, shape, dtype), bt


def _slots(bt, first, count):
    """Slots of positions first[b] .. first[b] + count[b] - 1 of every sequence."""
    out = []
    for b, (p0, n) in enumerate(zip(first, count)):
        p = torch.arange(p0, p0 + n)
        out.append(bt[b, p // PAGE].long() * PAGE + p % PAGE)
    return torch.cat(out).to(torch.int32)


def _cu(lens):
    c = torch.zeros(len(lens) + 1, dtype=torch.int32)
    c[1:] = torch.cumsum(torch.tensor(lens), 0)
    return c


def _qlinear(g, n, k, group, dtype):
    """An int8 linear as the loader leaves it: weights of standard deviation about 0.02."""
    lin = ReplicatedLinear(8, 8)
    w = torch.clamp(torch.round(torch.randn((n, k), generator=g, device="cuda") * 40), -127, 127).to(torch.int8)
    shape = (n, k // group) if group else (n,)
    s = ((torch.rand(shape, generator=g, device="cuda") + 0.5) * (0.02 / 40)).to(torch.bfloat16)
    lin.weight = torch.nn.Parameter(w, requires_grad=False)
    lin.weight_scale = torch.nn.Parameter(s, requires_grad=False)
    if group:
        lin.quant_granularity, lin.quant_group_size = "per_group", group
    return lin


def _norm(g, n, dtype):
    m = RMSNorm(n, EPS)
    m.weight = torch.nn.Parameter(1.0 + _randn(g, (n,), dtype, 0.1), requires_grad=False)
    return m


def _graphed(fn):
    """fn's work captured once, as the engine captures its decode steps; its outputs are static buffers."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


# ----------------------------------------------------------------------------------- attention
def _attn_meta(case):
    """(new rows, keys) per sequence."""
    lens = _case_lens(case)
    if case["kind"] == "decode":
        return [1] * len(lens), lens
    if case["kind"] == "verify":
        return [case["k"] + 1] * len(lens), [n + case["k"] for n in lens]
    return lens, [n + case.get("cached", 0) for n in lens]


def _prepare_attn(case, seed):
    g, cg = _gens(seed)
    dtype, hq = DTYPES[case["dtype"]], case["heads"]
    nq, nk = _attn_meta(case)
    kc, vc, bt = _pages(g, cg, nk, dtype)
    # q, k and v are the thirds of the qkv projection's output rows
    qkv = _randn(g, (sum(nq), (hq + 2 * KV_HEADS) * D), dtype)
    q, k, v = (t.unflatten(-1, (-1, D)) for t in qkv.split([hq * D, KV_HEADS * D, KV_HEADS * D], dim=-1))
    layer = Attention(hq, D, D ** -0.5, KV_HEADS)
    layer.k_cache, layer.v_cache = kc, vc
    slots = _slots(bt, [n - m for n, m in zip(nk, nq)], nq).cuda()
    bt_d = bt.cuda()
    if case["kind"] == "decode":
        ctx = dict(is_prefill=False, slot_mapping=slots, block_tables=bt_d,
                   context_lens=torch.tensor(nk, dtype=torch.int32).cuda())
    else:
        paged = case["kind"] == "verify" or case["cached"] > 0
        ctx = dict(is_prefill=True, cu_seqlens_q=_cu(nq).cuda(), cu_seqlens_k=_cu(nk).cuda(), max_seqlen_q=max(nq),
                   max_seqlen_k=max(nk), slot_mapping=slots, block_tables=bt_d if paged else None,
                   is_spec_verify=case["kind"] == "verify")
    return dict(layer=layer, q=q, k=k, v=v, ctx=ctx, bt=bt, slots=slots, nq=nq, nk=nk)


def _run_attn(s):
    set_context(**s["ctx"])
    return s["layer"](s["q"], s["k"], s["v"]), s["layer"].k_cache, s["layer"].v_cache


def _attend64(q, k, v):
    """Bottom-right causal attention in 64 bits: q (n, Hq, D), k / v (m, Hkv, D)."""
    n, hq, _ = q.shape
    m, hkv, _ = k.shape
    out = torch.empty_like(q)
    limit = torch.arange(m - n, m, device=q.device)[:, None]
    seen = torch.arange(m, device=q.device)[None, :] <= limit
    for h in range(hq):
        kv = h // (hq // hkv)
        s = (q[:, h] @ k[:, kv].T.contiguous()) * D ** -0.5
        s.masked_fill_(~seen, -math.inf)
        out[:, h] = torch.softmax(s, dim=-1) @ v[:, kv].contiguous()
    return out


def _exact_attn(case, seed):
    s = _prepare_attn(case, seed)
    kc, vc = s["layer"].k_cache.double(), s["layer"].v_cache.double()
    q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
    at = s["slots"].long()
    kc.view(-1, KV_HEADS, D)[at] = k
    vc.view(-1, KV_HEADS, D)[at] = v
    out, row = torch.empty_like(q), 0
    for b, (n, m) in enumerate(zip(s["nq"], s["nk"])):
        pos = _slots(s["bt"][b:b + 1], [0], [m]).long().cuda()
        out[row:row + n] = _attend64(q[row:row + n], kc.view(-1, KV_HEADS, D)[pos], vc.view(-1, KV_HEADS, D)[pos])
        row += n
    return out.unsqueeze(1) if case["kind"] == "decode" else out, kc, vc


def _work_attn(case):
    nq, nk = _attn_meta(case)
    hq = case.get("heads", SMALL["heads"])
    pairs = sum(n * m - n * (n - 1) // 2 for n, m in zip(nq, nk))
    kept = sum(nk) * KV_HEADS * D * 2 * 2           # every key and value once
    new = sum(nq) * KV_HEADS * D * 2 * 2            # the new rows into the pages
    return dict(bytes=kept + new + sum(nq) * hq * D * 2 * 2, flops=4.0 * pairs * hq * D)


# -------------------------------------------------------------------------------- linear blocks
def _dims(case):
    return SMALL if case.get("size", "small") == "small" else LARGE


def _prepare_mlp(case, seed):
    """RMSNorm with the residual add, gate_up, SiLU, down: a decoder layer's second half."""
    g, _ = _gens(seed)
    dtype, dim, m, group = DTYPES[case["dtype"]], _dims(case), case["rows"], case["group"]
    h, inter = dim["hidden"], dim["inter"]
    s = dict(norm=_norm(g, h, dtype), act=SiluAndMul(),
             gate_up=_qlinear(g, 2 * inter, h, group, dtype), down=_qlinear(g, h, inter, group, dtype),
             x=_randn(g, (m, h), dtype), res=_randn(g, (m, h), dtype))
    if m <= GRAPH_ROWS:
        if group:
            s["graph"], s["out"] = _graphed(lambda: _mlp(s))
        else:
            s["graph"], s["out"] = _graphed(lambda: _mlp_fused(s))
    return s


def _mlp(s):
    x, res = s["norm"](s["x"], s["res"])
    return s["down"](s["act"](s["gate_up"](x))), res


def _mlp_fused(s):
    """The draft step's form: the norm and the activation inside the projection."""
    res = torch.empty_like(s["res"])
    act = ops.w8a16_gate_up_silu(s["x"], s["gate_up"].weight, s["gate_up"].weight_scale, s["norm"].weight, EPS,
                                 residual=s["res"], residual_out=res)
    return ops.w8a16_linear(act, s["down"].weight, s["down"].weight_scale), res


def _run_mlp(s):
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    return _mlp(s)


def _weight64(lin):
    w, sc = lin.weight.double(), lin.weight_scale.double()
    if sc.dim() == 1:
        return w * sc[:, None]
    return (w.view(w.shape[0], sc.shape[1], -1) * sc[:, :, None]).view_as(w)


def _norm64(norm, x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * norm.weight.double()


def _mlp64(s, x, res):
    res = x + res
    gate, up = (_norm64(s["norm"], res) @ _weight64(s["gate_up"]).T).chunk(2, dim=-1)
    return (torch.nn.functional.silu(gate) * up) @ _weight64(s["down"]).T, res


def _exact_mlp(case, seed):
    s = _prepare_mlp(dict(case), seed)
    return _mlp64(s, s["x"].double(), s["res"].double())


def _linear_bytes(n, k, group):
    return n * k + 2 * n * (k // group if group else 1)


def _work_mlp(case):
    dim, m, group = _dims(case), case["rows"], case["group"]
    h, inter = dim["hidden"], dim["inter"]
    return dict(bytes=_linear_bytes(2 * inter, h, group) + _linear_bytes(h, inter, group) + 4 * m * h * 2 + 2 * h,
                flops=6.0 * m * h * inter)


def _prepare_head(case, seed):
    g, _ = _gens(seed)
    dtype, m, h = DTYPES[case["dtype"]], case["rows"], SMALL["hidden"]
    return dict(norm=_norm(g, h, dtype), lm=_qlinear(g, VOCAB, h, 0, dtype), x=_randn(g, (m, h), dtype),
                res=_randn(g, (m, h), dtype))


def _run_head(s):
    return ops.w8a16_rmsnorm_linear(s["x"], s["norm"].weight, EPS, s["lm"].weight, s["lm"].weight_scale,
                                    residual=s["res"])


def _exact_head(case, seed):
    s = _prepare_head(case, seed)
    return _norm64(s["norm"], s["x"].double() + s["res"].double()) @ _weight64(s["lm"]).T


def _work_head(case):
    m, h = case["rows"], SMALL["hidden"]
    return dict(bytes=_linear_bytes(VOCAB, h, 0) + 2 * m * h * 2 + 2 * h + m * VOCAB * 2, flops=2.0 * m * h * VOCAB)


# --------------------------------------------------------------------------------- decoder layer
def _rope_table(n):
    inv = 1.0 / (1e6 ** (torch.arange(0, D, 2, dtype=torch.float32, device="cuda") / D))
    a = torch.arange(n, dtype=torch.float32, device="cuda")[:, None] * inv[None, :]
    return torch.cat((a.cos(), a.sin()), dim=-1).contiguous()


def _prepare_layer(case, seed):
    g, cg = _gens(seed)
    dtype, hq, h, inter = DTYPES[case["dtype"]], SMALL["heads"], SMALL["hidden"], SMALL["inter"]
    lens = _case_lens(case)
    kc, vc, bt = _pages(g, cg, lens, dtype)
    attn = Attention(hq, D, D ** -0.5, KV_HEADS)
    attn.k_cache, attn.v_cache = kc, vc
    cu = _cu(lens).cuda()
    ctx = dict(is_prefill=True, cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=max(lens), max_seqlen_k=max(lens),
               slot_mapping=_slots(bt, [0] * len(lens), lens).cuda(), block_tables=None)
    return dict(lens=lens, attn=attn, ctx=ctx, in_norm=_norm(g, h, dtype), norm=_norm(g, h, dtype),
                q_norm=_norm(g, D, dtype).weight, k_norm=_norm(g, D, dtype).weight, act=SiluAndMul(),
                qkv=_qlinear(g, (hq + 2 * KV_HEADS) * D, h, 0, dtype), o=_qlinear(g, h, hq * D, 0, dtype),
                gate_up=_qlinear(g, 2 * inter, h, 0, dtype), down=_qlinear(g, h, inter, 0, dtype),
                pos=torch.cat([torch.arange(n) for n in lens]).cuda(), cos_sin=_rope_table(max(lens)),
                x=_randn(g, (sum(lens), h), dtype), res=_randn(g, (sum(lens), h), dtype))


def _run_layer(s):
    set_context(**s["ctx"])
    hq = SMALL["heads"]
    x, res = s["in_norm"](s["x"], s["res"])
    qkv = s["qkv"](x)
    q, k, v = (t.unflatten(-1, (-1, D)) for t in qkv.split([hq * D, KV_HEADS * D, KV_HEADS * D], dim=-1))
    ops.qk_norm_rope(q, k, s["pos"], s["cos_sin"], s["q_norm"], s["k_norm"], EPS)
    x = s["o"](s["attn"](q, k, v).flatten(1))
    x, res = s["norm"](x, res)
    return s["down"](s["act"](s["gate_up"](x))), res, s["attn"].k_cache, s["attn"].v_cache


def _exact_layer(case, seed):
    s = _prepare_layer(case, seed)
    hq, hkv = SMALL["heads"], KV_HEADS
    res = s["x"].double() + s["res"].double()
    qkv = _norm64(s["in_norm"], res) @ _weight64(s["qkv"]).T
    q, k, v = (t.unflatten(-1, (-1, D)) for t in qkv.split([hq * D, hkv * D, hkv * D], dim=-1))
    c, sn = (t[:, None, :] for t in s["cos_sin"].double()[s["pos"]].chunk(2, dim=-1))

    def rope(t, w):
        t = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + EPS) * w.double()
        a, b = t.chunk(2, dim=-1)
        return torch.cat((a * c - b * sn, b * c + a * sn), dim=-1)

    q, k = rope(q, s["q_norm"]), rope(k, s["k_norm"])
    kc, vc = s["attn"].k_cache.double(), s["attn"].v_cache.double()
    at = s["ctx"]["slot_mapping"].long()
    kc.view(-1, hkv, D)[at] = k
    vc.view(-1, hkv, D)[at] = v
    o, row = torch.empty_like(q), 0
    for n in s["lens"]:
        o[row:row + n] = _attend64(q[row:row + n], k[row:row + n], v[row:row + n])
        row += n
    out, res = _mlp64(s, o.flatten(1) @ _weight64(s["o"]).T, res)
    return out, res, kc, vc


def _work_layer(case):
    lens = _case_lens(case)
    t, h, inter, hq = sum(lens), SMALL["hidden"], SMALL["inter"], SMALL["heads"]
    shapes = [((hq + 2 * KV_HEADS) * D, h), (h, hq * D), (2 * inter, h), (h, inter)]
    pairs = sum(n * (n + 1) // 2 for n in lens)
    return dict(bytes=sum(_linear_bytes(n, k, 0) for n, k in shapes) + 4 * t * h * 2 + t * KV_HEADS * D * 2 * 2,
                flops=2.0 * t * sum(n * k for n, k in shapes) + 4.0 * pairs * hq * D)


# ------------------------------------------------------------------------------------ draft model
def _prepare_draft(case, seed):
    """The draft model with a prefilled context, its decode step captured in a graph."""
    chain = DraftChain(case["batch"], ctx_len=case["ctx"], k=1, layers=LAYERS, seed=seed, fused=True)
    graph, logits = _graphed(lambda: chain.step(0))
    return dict(chain=chain, graph=graph, logits=logits)


def _run_draft(s):
    s["graph"].replay()
    return s["logits"]


def _work_draft(case):
    b, h, inter, hq = case["batch"], SMALL["hidden"], SMALL["inter"], SMALL["heads"]
    shapes = [((hq + 2 * KV_HEADS) * D, h), (h, hq * D), (2 * inter, h), (h, inter)]
    weights = LAYERS * sum(_linear_bytes(n, k, 0) for n, k in shapes) + _linear_bytes(VOCAB, h, 0)
    kv = LAYERS * b * (case["ctx"] + 2) * KV_HEADS * D * 2 * 2
    return dict(bytes=weights + kv + b * h * 2 + b * VOCAB * 2,
                flops=2.0 * b * (LAYERS * sum(n * k for n, k in shapes) + VOCAB * h)
                + 4.0 * LAYERS * b * (case["ctx"] + 1) * hq * D)


# ---------------------------------------------------------------------------------- verification
def _prepare_accept(case, seed):
    """Target logits, and a draft that agrees with them in part; tokens drawn from the draft."""
    g, _ = _gens(seed)
    b, k, dtype = case["batch"], case["k"], DTYPES[case["dtype"]]
    target = torch.randn((b, k + 1, VOCAB), generator=g, device="cuda") * 2.5
    draft = target[:, :k] + torch.randn((b, k, VOCAB), generator=g, device="cuda") * 0.5
    temps = torch.rand((b,), generator=g, device="cuda") * 0.5 + 0.6
    noise = torch.empty((b, k, VOCAB), device="cuda").exponential_(generator=g)
    tokens = (draft / temps[:, None, None] - noise.log()).argmax(-1)
    return dict(draft=draft.to(dtype), target=target.to(dtype), tokens=tokens, temps=temps,
                rng=torch.tensor([seed, 17], dtype=torch.int64, device="cuda"))


def _run_accept(s):
    r = verify_batch(s["draft"], s["target"], s["tokens"], s["temps"], rng_state=s["rng"])
    return r.accepted, r.bonus, r.accept_mask


def _work_accept(case):
    rows = case["batch"] * (2 * case["k"] + 1)
    return dict(bytes=rows * VOCAB * (4 if case["dtype"] == "fp32" else 2), flops=4.0 * rows * VOCAB)


# --------------------------------------------------------------------------------------- entries
_PREPARE = dict(draft=_prepare_draft, decode=_prepare_attn, verify=_prepare_attn, prefill=_prepare_attn,
                layer=_prepare_layer, mlp=_prepare_mlp, head=_prepare_head, accept=_prepare_accept)
_RUN = dict(draft=_run_draft, decode=_run_attn, verify=_run_attn, prefill=_run_attn, layer=_run_layer,
            mlp=_run_mlp, head=_run_head, accept=_run_accept)
_WORK = dict(draft=_work_draft, decode=_work_attn, verify=_work_attn, prefill=_work_attn, layer=_work_layer,
             mlp=_work_mlp, head=_work_head, accept=_work_accept)
_EXACT = dict(decode=_exact_attn, verify=_exact_attn, prefill=_exact_attn, layer=_exact_layer, mlp=_exact_mlp,
              head=_exact_head)


def prepare(case, seed):
    with torch.no_grad():
        state = _PREPARE[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


def run(state):
    with torch.no_grad():
        return _RUN[state["kind"]](state)


def work(case):
    return _WORK[case["kind"]](case)


def exact(case, seed):
    """The result in 64 bits; None for the 28-layer model (bf16 rounding between its layers, not the sums
    inside them, decides its logits) and for the verification, whose results are whole numbers."""
    if case["kind"] not in _EXACT:
        return None
    with torch.no_grad():
        return _EXACT[case["kind"]](case, seed)


# (rel, max) in bf16: four times the distance from the 64-bit result, measured over the listed cases of each kind
# (16-bit rounding of the outputs and, in the blocks, of what passes between the layers); fp16 has 3 bits more.
_TOLERANCE = dict(decode=(0.007, 0.016), verify=(0.007, 0.016), prefill=(0.009, 0.045), layer=(0.023, 0.15),
                  mlp=(0.02, 0.13), head=(0.012, 0.07))


def tolerance(case):
    if case["kind"] == "accept":
        return "exact"
    if case["kind"] == "draft":
        # the fused and the unfused step of this library are 0.012 (largest 0.063) apart at 16 sequences: a
        # rounding that falls the other way in one layer travels through all that follow
        return {"rel": 0.03, "max": 0.25}
    rel, most = _TOLERANCE[case["kind"]]
    unit = 1 if case["dtype"] == "bf16" else 8
    return {"rel": rel / unit, "max": most / unit}
