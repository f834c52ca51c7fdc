"""The work that is timed: one pass each of what a user of this framework has it do.

The model is the repository's own Qwen3-1.7B shape (hidden 2048, intermediate 6144, 16 query and 8 kv
heads of 128, an 8192-token SID head).  Serving it means: prefill of one or several prompts, then a few
decode steps over requests x beams rows (20 beams of one request up to 8 requests of 512 beams), each
step ending in the SID head and the trie-constrained beam selection.  Decode runs inside HIP graphs, as
``Qwen3FP8DecodeStep.capture`` records it; prefill and the head's log-probabilities run eagerly.
"""

import math
from types import SimpleNamespace

import torch

from flashrec_amd.attention import AttentionBackend
from flashrec_amd.decode_step import Qwen3FP8DecodeStep, Qwen3Shape
from flashrec_amd.kernel.beam_trie import GenrecFusedWorkspace, genrec_mask_topk_expand, row_topk
from flashrec_amd.kernel.qk_rope_kv import fused_qk_norm_rope_store_fp8
from flashrec_amd.kernel.sglops import per_token_quant_fp8
from flashrec_amd.kernel.silu_fp8 import silu_and_mul_per_token_quant_fp8
from flashrec_amd.kvcache.pool import TokenToKVPool
from flashrec_amd.layers.linear import Linear
from flashrec_amd.layers.norm import RMSNorm
from flashrec_amd.layers.rotary import RotaryEmbedding
from flashrec_amd.logits import RestrictedLMHead

HIDDEN, INTER, HQ, HK, D, SID = 2048, 6144, 16, 8, 128, 8192
EPS, THETA, MAX_POS = 1e-6, 1e6, 4096
LEVELS, CODES, ITEMS = 3, 256, 65536


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the MLP of a decode step: one request at the narrowest beam served, one
        # at a wide beam, and a full batch of 8 wide requests
        {"name": "mlp-20", "kind": "mlp", "rows": 20},
        {"name": "mlp-512", "kind": "mlp", "rows": 512},
        {"name": "mlp-4096", "kind": "mlp", "rows": 4096},
        # the attention block of a decode step: one request with a short prompt,
        # one with a long user history, the full batch
        {"name": "attn-1x50", "kind": "attn", "requests": 1, "beams": 50, "prefix": 200, "step": 1},
        {"name": "attn-1x512-long", "kind": "attn", "requests": 1, "beams": 512, "prefix": 1500, "step": 2},
        {"name": "attn-8x512", "kind": "attn", "requests": 8, "beams": 512, "prefix": 128, "step": 1},
        # the attention block of a prefill: one long prompt, and a batch of
        # short ragged ones whose first tokens are in the prefix cache
        {"name": "prefill-1x1999", "kind": "prefill", "requests": 1, "tokens": 1999, "cached": 0},
        {"name": "prefill-8x256", "kind": "prefill", "requests": 8, "tokens": 256, "cached": 37},
        # the MLP through the drop-in operators one by one (a reference user
        # who changed only the imports), an odd number of prefill rows
        {"name": "dropin-1001", "kind": "dropin", "rows": 1001, "dtype": "bf16"},
        # the end of a step: the restricted head's log-probabilities, and the
        # head with the beam selection of the full batch
        {"name": "logprobs-128", "kind": "logprobs", "rows": 128},
        {"name": "beam-8x512", "kind": "beam", "requests": 8, "beams": 512},
        # a whole decode step of the full batch
        {"name": "step-8x512", "kind": "step", "requests": 8, "beams": 512, "prefix": 128, "step": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "attn", "attn", "prefill", "prefill", "dropin", "logprobs", "beam", "step"])
    if kind in ("mlp", "logprobs"):
        return {"kind": kind, "rows": _log(rng, 1 if kind == "mlp" else 8, 4096)}
    if kind == "dropin":
        return {"kind": kind, "rows": _log(rng, 8, 4096), "dtype": rng.choice(["bf16", "bf16", "bf16", "fp16"])}
    if kind == "prefill":
        requests = rng.choice([1, 1, 2, 4, 8])
        tokens = _log(rng, 24, 4000 // requests)
        return {"kind": kind, "requests": requests, "tokens": tokens,
                "cached": rng.choice([0, 0, rng.randrange(1, tokens // 2 + 1)])}
    requests, beams = rng.choice([1, 1, 2, 3, 4, 8]), _log(rng, 20, 512)
    if kind == "beam":
        return {"kind": kind, "requests": requests, "beams": beams}
    # whole steps stay below the cost of the listed one
    prefix = _log(rng, 48, 3000 if kind == "attn" else min(600, 48 + 300000 // (requests * beams)))
    return {"kind": kind, "requests": requests, "beams": beams, "prefix": prefix, "step": rng.randrange(1, 4)}


# ------------------------------------------------------------------ inputs
# Every tensor comes from a generator of its own (the case's seed and the
# tensor's number), so that exact() makes the same ones again without the package.
def _randn(seed, number, *shape):
    g = torch.Generator(device="cuda").manual_seed(1000 * int(seed) + number)
    return torch.randn(*shape, generator=g, device="cuda")


def _dtype(case):
    return torch.float16 if case.get("dtype") == "fp16" else torch.bfloat16


def _rows_in(seed, number, rows, dtype=torch.bfloat16):
    """Hidden rows: N(0, 1) with 1 % of the channels x20 (the outlier channels of decoder activations)."""
    x = _randn(seed, number, rows, HIDDEN)
    x[:, 7::100] *= 20.0
    return x.to(dtype)


def _weight(seed, number, n, k):
    return (0.02 * _randn(seed, number, n, k)).to(torch.bfloat16)


def _gamma(seed, number, n):
    return (1.0 + 0.1 * _randn(seed, number, n)).to(torch.bfloat16)


def _linear(seed, number, n, k):
    lin = Linear(k, n)
    lin.load(_weight(seed, number, n, k), quantize_fp8=True)
    lin.prepare()
    return lin


def _norm(seed, number, n):
    norm = RMSNorm(n, EPS)
    norm.weight = torch.nn.Parameter(_gamma(seed, number, n), requires_grad=False)
    return norm


def _prompts(case):
    """(tokens in the prefix cache, new tokens) of each prompt of a prefill."""
    out = []
    for i in range(case["requests"]):
        total = max(2, case["tokens"] - (i * 89) % (case["tokens"] * 3 // 4))
        cached = min(case["cached"], total - 1)
        out.append((cached, total - cached))
    return out


def _layout(case, seed):
    """Slots, positions and row bounds of a decode or prefill batch: slots in the
    order of a pool that has been in use (a permutation; slot 0 is the dummy)."""
    g = torch.Generator().manual_seed(1000 * int(seed) + 999)
    if case["kind"] == "attn":
        n, bw, prefix, own = case["requests"], case["beams"], case["prefix"], case["step"] + 1
        rows, slots = n * bw, 1 + n * prefix + n * bw * own
        perm = (1 + torch.randperm(slots - 1, generator=g)).to(torch.int32)
        shared = perm[:n * prefix].view(n, prefix)
        mine = perm[n * prefix:].view(rows, own)
        kv = torch.cat([shared[torch.arange(rows) // bw], mine], dim=1)
        return SimpleNamespace(slots=slots, rows=rows, kv=kv, lens=torch.full((rows,), prefix + own, dtype=torch.int32),
                               positions=torch.full((rows,), prefix + own - 1), loc=mine[:, -1].long())
    prompts = _prompts(case)
    total = sum(c + e for c, e in prompts)
    perm = (1 + torch.randperm(total, generator=g)).to(torch.int32)
    loc, pos, at = [], [], 0
    for c, e in prompts:
        loc.append(perm[at + c:at + c + e].long())
        pos.append(torch.arange(c, c + e))
        at += c + e
    return SimpleNamespace(slots=1 + total, rows=sum(e for _, e in prompts), kv=perm, prompts=prompts,
                           lens=torch.tensor([c + e for c, e in prompts], dtype=torch.int32),
                           positions=torch.cat(pos), loc=torch.cat(loc))


def _caches(seed, slots):
    k = _randn(seed, 30, slots, HK, D)
    v = _randn(seed, 31, slots, HK, D)
    return k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)


def _trie(seed):
    """A random trie of 3-code items as dense tables (allow, next node), and its first-level codes."""
    g = torch.Generator(device="cuda").manual_seed(1000 * int(seed) + 40)
    sids = torch.randint(0, CODES, (ITEMS, LEVELS), generator=g, device="cuda")
    nodes, count, key = [torch.zeros(ITEMS, dtype=torch.int64, device="cuda")], 1, torch.zeros_like(sids[:, 0])
    for d in range(1, LEVELS):
        key = key * CODES + sids[:, d - 1]
        uniq, inverse = torch.unique(key, return_inverse=True)
        nodes.append(count + inverse)
        count += int(uniq.numel())
    allow = torch.zeros(count + 1, LEVELS * CODES, dtype=torch.bool, device="cuda")
    nxt = torch.full((count + 1, LEVELS * CODES), count, dtype=torch.int32, device="cuda")
    for d in range(LEVELS):
        rel = d * CODES + sids[:, d]
        allow[nodes[d], rel] = True
        nxt[nodes[d], rel] = nodes[d + 1].to(torch.int32) if d + 1 < LEVELS else -1
    return allow, nxt, count, sids


def _captured(state, one):
    """Record ``one(state)`` into a HIP graph after a warm-up, as a serving loop does per batch shape."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        one(state)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        state["out"] = one(state)
    state["graph"] = graph
    return state


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind}
    if kind in ("mlp", "dropin"):
        state["x"] = _rows_in(seed, 1, case["rows"], _dtype(case))
        state["norm"] = _norm(seed, 10, HIDDEN)
        state["gate_up"], state["down"] = _linear(seed, 11, 2 * INTER, HIDDEN), _linear(seed, 12, HIDDEN, INTER)
        if kind == "dropin":
            state["hidden"] = _randn(seed, 2, case["rows"], HIDDEN).to(_dtype(case))
            state["dtype"] = _dtype(case)
            return state
        state["gate_up"]._glu_operands()
        return _captured(state, _mlp)
    if kind in ("attn", "prefill"):
        lay = _layout(case, seed)
        state["x"] = _rows_in(seed, 1, lay.rows)
        state["norm"], state["q_norm"], state["k_norm"] = (_norm(seed, 10 + i, n) for i, n in enumerate((HIDDEN, D, D)))
        state["qkv"], state["o"] = _linear(seed, 20, (HQ + 2 * HK) * D, HIDDEN), _linear(seed, 21, HIDDEN, HQ * D)
        state["rotary"] = RotaryEmbedding(D, MAX_POS, THETA, device="cuda")
        pool = TokenToKVPool(1, lay.slots, HK, D, torch.float8_e4m3fn, torch.device("cuda"))
        for cache, values in zip((pool.k[0], pool.v[0]), _caches(seed, lay.slots)):
            cache.copy_(values)
        prefill = kind == "prefill"
        batch = SimpleNamespace(is_prefill=prefill, n_rows=int(lay.lens.numel()), seq_lens=lay.lens.cuda(),
                                seq_lens_cpu=lay.lens, kv_indices=lay.kv.reshape(-1).cuda(), kv_indptr=None,
                                positions=lay.positions.cuda(), out_cache_loc=lay.loc.cuda(),
                                extend_seq_lens=[e for _, e in lay.prompts] if prefill else None,
                                extend_prefix_lens=[c for c, _ in lay.prompts] if prefill else None)
        state["pool"], state["batch"] = pool, batch
        state["attention"] = AttentionBackend(pool, HQ, HK, D)
        state["attention"].prepare(batch)
        return state if prefill else _captured(state, _attn)
    if kind == "step":
        shape = Qwen3Shape()
        state["step"] = Qwen3FP8DecodeStep(shape, case["requests"], case["beams"], case["prefix"], case["step"],
                                           seed=int(seed))
        state["step"].capture()
        return state
    # the head: a bf16 lm_head whose top rows are the SID tokens
    rows = case["rows"] if kind == "logprobs" else case["requests"] * case["beams"]
    state["x"] = _rows_in(seed, 1, rows)
    state["lm"] = _weight(seed, 20, SID, HIDDEN)
    state["head"] = RestrictedLMHead(list(range(SID)), fp8=True)
    state["head"].bind(state["lm"])
    if kind == "logprobs":
        return state
    n, bw = case["requests"], case["beams"]
    state["norm"] = _norm(seed, 10, HIDDEN)
    state["allow"], state["next"], state["invalid"], sids = _trie(seed)
    g = torch.Generator(device="cuda").manual_seed(1000 * int(seed) + 41)
    first = sids[torch.randint(0, ITEMS, (n, bw), generator=g, device="cuda"), 0]
    state["n"], state["bw"], state["c"] = n, bw, 2 * bw
    state["ids"] = torch.arange(SID, dtype=torch.int64, device="cuda")
    state["cum"] = torch.sort(_randn(seed, 42, n, bw) - 3.0, dim=-1, descending=True).values
    state["nodes"] = state["next"][0, first].to(torch.int64)
    state["tokens"] = torch.zeros(n, bw, LEVELS, dtype=torch.int64, device="cuda")
    state["tokens"][:, :, 0] = first
    state["col"] = torch.ones(n, dtype=torch.int32, device="cuda")
    state["workspace"] = GenrecFusedWorkspace()
    return _captured(state, _beam)


# ------------------------------------------------------------------ one pass
def _mlp(s):
    x = s["x"].clone()  # the residual stream is updated in place
    q, a = s["norm"].quant_fp8(x)
    y = s["gate_up"].forward_fp8_silu(q, a)
    return s["down"].forward_fp8_residual(*per_token_quant_fp8(y), x)


def _qkv(s, q, a):
    t = q.shape[0]
    heads = s["qkv"].forward_fp8(q, a, (t, HIDDEN), torch.bfloat16).view(t, HQ + 2 * HK, D)
    qh, kh, vh = heads[:, :HQ], heads[:, HQ:HQ + HK], heads[:, HQ + HK:]
    b, pool = s["batch"], s["pool"]
    if not fused_qk_norm_rope_store_fp8(qh, kh, vh, b.positions, b.out_cache_loc, s["q_norm"].weight,
                                        s["k_norm"].weight, EPS, s["rotary"].cos_sin_cache, pool.k[0], pool.v[0]):
        raise RuntimeError("the fused QK-norm / RoPE / KV write did not run")
    return qh, kh, vh


def _attn(s):
    x = s["x"].clone()  # the residual stream is updated in place
    qh, _, _ = _qkv(s, *s["norm"].quant_fp8(x))
    x = s["o"].forward_fp8_residual(*s["attention"].forward_quant_fp8(qh, 0), x)
    return x, s["pool"].k[0], s["pool"].v[0]


def _beam(s):
    logits, _ = s["head"].compute_logits_fp8(*s["norm"].quant_fp8(s["x"]), s["lm"])
    vals, _, toks = row_topk(logits.view(s["n"], s["bw"], -1), s["c"], s["ids"], need_idx=False, log_softmax=True)
    r = genrec_mask_topk_expand(s["cum"], vals, toks, select_k=s["bw"], node_ids=s["nodes"], allow_table=s["allow"],
                                token_base=0, token_ids=s["tokens"], col=s["col"], next_node=s["next"],
                                invalid_node=s["invalid"], workspace=s["workspace"])
    return logits, vals, toks, r.vals, r.parents, r.tokens, r.token_ids, r.node_ids


def run(state):
    kind = state["kind"]
    if kind == "step":
        return state["step"].replay()
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if kind == "prefill":
        x = state["x"]
        qh, kh, vh = _qkv(state, *state["norm"].quant_fp8(x))
        o = state["attention"].forward(qh, kh, vh, 0, state["batch"], skip_store=True)
        return state["o"](o.reshape(x.shape[0], -1)), state["pool"].k[0], state["pool"].v[0]
    if kind == "dropin":
        residual = state["x"].clone()  # updated in place by the fused add
        q, a, residual = state["norm"].quant_fp8(state["hidden"], residual)
        gu = state["gate_up"].forward_fp8(q, a, tuple(residual.shape), state["dtype"])
        q, a = silu_and_mul_per_token_quant_fp8(gu)
        return state["down"].forward_fp8(q, a, (q.shape[0], INTER), state["dtype"]), residual
    return state["head"].compute(state["x"], state["lm"])[0]


# ------------------------------------------------------------------ what a pass cannot do without
def _gemm(rows, n, k):
    return n * k + 4 * n, 2 * rows * n * k


def work(case):
    kind = case["kind"]
    if kind in ("mlp", "dropin"):
        m = case["rows"]
        parts = [_gemm(m, 2 * INTER, HIDDEN), _gemm(m, HIDDEN, INTER)]
        io = (4 if kind == "mlp" else 8) * m * HIDDEN  # x (hidden, residual) in, residual (and output) out
    elif kind in ("attn", "prefill"):
        if kind == "attn":
            m = case["requests"] * case["beams"]
            seen = m * (case["prefix"] + case["step"] + 1)
            slots = case["requests"] * case["prefix"] + m * (case["step"] + 1)
        else:
            prompts = _prompts(case)
            m, slots = sum(e for _, e in prompts), sum(c + e for c, e in prompts)
            seen = sum(c * e + e * (e + 1) // 2 for c, e in prompts)
        parts = [_gemm(m, (HQ + 2 * HK) * D, HIDDEN), _gemm(m, HIDDEN, HQ * D),
                 (slots * 2 * HK * D, 4 * HQ * D * seen)]
        io = 4 * m * HIDDEN + 4 * seen // (m if kind == "prefill" else 1) + 24 * m
    elif kind == "step":
        m = case["requests"] * case["beams"]
        layers = 28
        seen = m * (case["prefix"] + case["step"] + 1)
        slots = case["requests"] * case["prefix"] + m * (case["step"] + 1)
        one = [_gemm(m, (HQ + 2 * HK) * D, HIDDEN), _gemm(m, HIDDEN, HQ * D), _gemm(m, 2 * INTER, HIDDEN),
               _gemm(m, HIDDEN, INTER), (slots * 2 * HK * D, 4 * HQ * D * seen)]
        parts = one * layers + [_gemm(m, SID, HIDDEN)]
        io = 2 * m * HIDDEN + 4 * m * SID
    else:
        m = case["rows"] if kind == "logprobs" else case["requests"] * case["beams"]
        parts = [_gemm(m, SID, HIDDEN)]
        io = 2 * m * HIDDEN + 4 * m * SID
        if kind == "beam":  # the top 2 * beams (value, token) of each row, the selected beams
            io += m * 2 * case["beams"] * 12 + m * (8 * LEVELS * 2 + 40)
    return {"bytes": float(io + sum(b for b, _ in parts)), "flops": float(sum(f for _, f in parts))}


def tolerance(case):
    """About three to four times the largest distance seen from exact() (in
    parentheses), which is what another rounding of the same sums does: a
    16-bit rounding that falls the other way moves an e4m3 code by 2^-4 of its
    value, and the codes feed the next product.  The step: measured against
    itself with the attention's probabilities kept in fp32 (0.018)."""
    return {"mlp": {"rel": 2e-2},        # (0.0057)
            "attn": {"rel": 2e-2},       # (0.0057, the stored K rows)
            "prefill": {"rel": 7e-2},    # (0.023: the o projection's codes, after bf16 probabilities)
            "dropin": {"rel": 4e-2},     # (0.012)
            "logprobs": {"rel": 2e-3},   # (0.00057)
            # (0.0035); neighbours in the top-k order swap where logits nearly tie
            "beam": {"rel": 1.2e-2, "differ": 2e-2},
            "step": {"rel": 6e-2}}[case["kind"]]


# ------------------------------------------------------------------ the same in 64 bits
# Plain torch in float64; values are rounded where an operator's result is a
# 16-bit or e4m3 tensor by definition (codes, scales, bf16 rows), nowhere else.
def _quant(x):
    amax = x.abs().amax(-1, keepdim=True).clamp(min=1e-12)
    scale = (amax.float() / 448.0)
    codes = (x.float() / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return codes.double(), scale.double()


def _mm(codes, scale, seed, number, n, k):
    w, ws = _quant(_weight(seed, number, n, k).double())
    return (codes @ w.t()) * scale * ws.t()


def _rms(x, gamma, dtype):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return (y * gamma.to(dtype).double()).to(dtype).double()


def _exact_attention(case, seed, lay, q, kc, vc):
    """Softmax attention of each row over its own slots, float64."""
    scale, out = D ** -0.5, torch.empty_like(q)
    if case["kind"] == "attn":
        kv = lay.kv.long().cuda()
        for a in range(0, lay.rows, 128):
            slots = kv[a:a + 128]
            k = kc[slots].repeat_interleave(HQ // HK, dim=2)  # [rows, keys, heads, dims]
            p = torch.softmax((q[a:a + 128, None] * k).sum(-1) * scale, dim=1)
            out[a:a + 128] = (p[..., None] * vc[slots].repeat_interleave(HQ // HK, dim=2)).sum(1)
        return out
    at = row = 0
    for c, e in lay.prompts:
        slots = lay.kv[at:at + c + e].long().cuda()
        mask = torch.arange(c + e, device="cuda")[None] > torch.arange(c, c + e, device="cuda")[:, None]
        for h in range(HQ):
            s = (q[row:row + e, h] @ kc[slots, h * HK // HQ].t()) * scale
            out[row:row + e, h] = torch.softmax(s.masked_fill(mask, -math.inf), dim=1) @ vc[slots, h * HK // HQ]
        at, row = at + c + e, row + e
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return None
    if kind in ("mlp", "dropin"):
        dt = _dtype(case)
        x = _rows_in(seed, 1, case["rows"], dt).double()
        if kind == "dropin":
            x = (x + _randn(seed, 2, case["rows"], HIDDEN).to(dt).double()).to(dt).double()
        gu = _mm(*_quant(_rms(x, _gamma(seed, 10, HIDDEN), dt)), seed, 11, 2 * INTER, HIDDEN).to(dt).double()
        g, u = gu[:, :INTER], gu[:, INTER:]
        y = ((g / (1.0 + torch.exp(-g))).to(dt).double() * u).to(dt).double()
        out = _mm(*_quant(y), seed, 12, HIDDEN, INTER).to(dt)
        return (out.double() + x).to(dt) if kind == "mlp" else (out, x.to(dt))
    if kind in ("attn", "prefill"):
        bf, lay = torch.bfloat16, _layout(case, seed)
        x = _rows_in(seed, 1, lay.rows).double()
        qkv = _mm(*_quant(_rms(x, _gamma(seed, 10, HIDDEN), bf)), seed, 20, (HQ + 2 * HK) * D, HIDDEN)
        heads = qkv.to(bf).double().view(lay.rows, HQ + 2 * HK, D)
        inv = 1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
        ang = torch.outer(torch.arange(MAX_POS, dtype=torch.float32), inv)
        cos, sin = (f(ang)[lay.positions].double().cuda()[:, None].repeat(1, 1, 2) for f in (torch.cos, torch.sin))
        turned = []
        for h, number in ((heads[:, :HQ], 11), (heads[:, HQ:HQ + HK], 12)):
            h = _rms(h, _gamma(seed, number, D), bf)
            half = torch.cat([-h[..., D // 2:], h[..., :D // 2]], dim=-1)
            turned.append((h * cos + half * sin).to(bf).double())
        kc, vc = (c.double() for c in _caches(seed, lay.slots))
        loc = lay.loc.cuda()
        kc[loc] = turned[1].float().to(torch.float8_e4m3fn).double()
        vc[loc] = heads[:, HQ + HK:].float().to(torch.float8_e4m3fn).double()
        o = _exact_attention(case, seed, lay, turned[0], kc, vc).to(bf).double().view(lay.rows, HQ * D)
        out = _mm(*_quant(o), seed, 21, HIDDEN, HQ * D).to(bf)
        return ((out.double() + x).to(bf) if kind == "attn" else out), kc, vc
    rows = case["rows"] if kind == "logprobs" else case["requests"] * case["beams"]
    x = _rows_in(seed, 1, rows).double()
    if kind == "beam":
        x = _rms(x, _gamma(seed, 10, HIDDEN), torch.bfloat16)
    logits = _mm(*_quant(x), seed, 20, SID, HIDDEN)
    lp = torch.log_softmax(logits, dim=-1)
    if kind == "logprobs":
        return lp
    n, bw = case["requests"], case["beams"]
    vals = torch.sort(lp, dim=-1, descending=True).values
    return logits, vals[:, :2 * bw].reshape(n, bw, -1), None, None, None, None, None, None
