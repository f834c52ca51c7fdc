"""Attention plans read by calls they were not made for exactly: a plan of
more tokens, graph decode with fewer rows than were captured, buffers of zeros
and of bare prefixes, each against the fp32 oracle."""

import pytest
import torch

from oracle import ops

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn
SCALE = 128 ** -0.5
# a probability rounded to bf16 moves a row by at most 2^-9 max |v| (|v| < 5),
# the output's own rounding by 2^-9 of it
BOUND = 2.0 ** -9 * 5 + 2.0 ** -8 * 5


def _inputs(dev, hq, hk, seed=3):
    """88 tokens: three requests of odd beam counts over prompts of 40, 200 and
    8 slots, 2 own slots each, and a causal prompt of 30 tokens."""
    g = torch.Generator().manual_seed(seed)
    perm = (1 + torch.randperm(1000, generator=g)).to(torch.int32)
    lists, lens, at = [], [], 0
    for prefix, beams in ((40, 21), (200, 30), (8, 7)):
        head, at = perm[at:at + prefix], at + prefix
        for _ in range(beams):
            lists.append(torch.cat([head, perm[at:at + 2]]))
            lens.append(prefix + 2)
            at += 2
    start = [0]
    for x in lists:
        start.append(start[-1] + x.numel())
    lists.append(perm[at:at + 30])
    start = start[:-1] + [start[-1]] * 30
    lens += list(range(1, 31))
    k = torch.randn(1001, hk, 128, generator=g).to(E4M3)
    v = torch.randn(1001, hk, 128, generator=g).to(E4M3)
    q = torch.randn(len(lens), hq, 128, generator=g).to(torch.bfloat16)
    return [x.to(dev) for x in (q, k, v, torch.cat(lists), torch.tensor(start, dtype=torch.int32),
                                torch.tensor(lens, dtype=torch.int32))]


@pytest.mark.parametrize("hq,hk", [(16, 8), (8, 8), (16, 4), (16, 2)])
def test_plan_of_other_token_counts(dev, hq, hk):
    from flashrec_amd.attention import attention_plan, paged_attention, paged_attention_quant_fp8, plan_size
    from flashrec_amd.kernel.sglops import per_token_quant_fp8

    q, k, v, idx, start, ln = _inputs(dev, hq, hk)
    n = int(ln.numel())
    plan = attention_plan(idx, start, ln, hq, hk)
    flat = torch.zeros(plan_size(n, hq, hk) + 5, dtype=torch.int32, device=dev)
    assert torch.equal(attention_plan(idx, start, ln, hq, hk, out=flat), plan)
    bare = torch.full((plan.numel() + 3,), -1, dtype=torch.int32, device=dev)
    assert attention_plan(idx, start, ln, hq, hk, out=bare) is bare
    assert torch.equal(bare[:-3], plan) and bool((bare[-3:] == -1).all())
    zero, shifted = torch.zeros_like(flat), plan[1:]
    want = ops.paged_attention(*(x.cpu() for x in (q, k, v, idx, start, ln)), SCALE).float()
    for t in (1, 15, 16, 17, 40, 48, 64, 80, n - 1, n):
        print(f"plan of {n} read by {t}, {hq}/{hk}", flush=True)
        tok = 32 * hk // hq
        plans = [plan, flat, bare, zero, zero[: plan.numel()]]
        if -(-t // tok) < plan.numel():
            plans.append(shifted)  # another group's records are no plan of this one
        for i, gp in enumerate(plans):
            got = paged_attention(q[:t], k, v, idx, start, ln, SCALE, group_prefix=gp)
            assert (got.float().cpu() - want[:t]).abs().max().item() < BOUND, (t, i)
            codes, s = paged_attention_quant_fp8(q[:t], k, v, idx, start, ln, SCALE, group_prefix=gp)
            ref, ref_s = per_token_quant_fp8(got.reshape(t, hq * 128))
            assert torch.equal(codes.view(torch.uint8), ref.view(torch.uint8)) and torch.equal(s, ref_s), (t, i)


@pytest.mark.parametrize("waves", [1, 4])
def test_tokens_past_the_plan(dev, waves):
    """A call of more tokens than the plan knows (the padding rows of a captured
    launch): the known ones are right, the others come out finite."""
    from flashrec_amd._lib import call
    from flashrec_amd.attention import attention_plan, plan_size

    hq, hk = 16, 8
    q, k, v, idx, start, ln = _inputs(dev, hq, hk)
    want = ops.paged_attention(*(x.cpu() for x in (q, k, v, idx, start, ln)), SCALE).float()
    t = int(ln.numel())
    for known in (1, 5, 21, 32, 50, 60, 87):
        print(f"plan of {known} read by {t}, waves {waves}", flush=True)
        plan = torch.zeros(plan_size(t, hq, hk), dtype=torch.int32, device=dev)
        attention_plan(idx, start[:known], ln[:known], hq, hk, out=plan)
        out = torch.full((t, hq, 128), float("nan"), dtype=torch.bfloat16, device=dev)
        call("fr_paged_attention_split_fp8", q.data_ptr(), hq * 128, 128, k.data_ptr(), hk * 128, 128, v.data_ptr(),
             hk * 128, 128, k.shape[0], idx.data_ptr(), start.data_ptr(), ln.data_ptr(), out.data_ptr(), hq * 128,
             128, t, hq, hk, 128, SCALE, plan.data_ptr(), waves, torch.cuda.current_stream().cuda_stream)
        got = out.float().cpu()
        assert bool(torch.isfinite(got).all())
        assert (got[:known] - want[:known]).abs().max().item() < BOUND


@pytest.mark.parametrize("quant", [False, True])
def test_graph_decode_of_fewer_rows(dev, quant):
    """Rows 0 .. n - 1 of a graph captured with bs rows, over batches of fewer."""
    from types import SimpleNamespace

    from flashrec_amd.attention import AttentionBackend
    from flashrec_amd.kvcache.pool import TokenToKVPool

    hq, hk, slots, bs, maxlen = 16, 8, 1024, 40, 150
    g = torch.Generator().manual_seed(9)
    pool = TokenToKVPool(1, slots, hk, 128, E4M3, dev)
    k0 = torch.randn(slots, hk, 128, generator=g).to(E4M3)
    v0 = torch.randn(slots, hk, 128, generator=g).to(E4M3)
    pool.k_cache(0).copy_(k0.to(dev))
    pool.v_cache(0).copy_(v0.to(dev))
    be = AttentionBackend(pool, hq, hk, 128)
    be.init_graph_wrappers([bs], maxlen)
    be.begin_graph_decode(bs)
    q = torch.randn(bs, hq, 128, generator=g).to(torch.bfloat16).to(dev)

    def batch(n, shared):
        head = torch.randint(1, slots, (shared,), generator=g, dtype=torch.int32)
        lists = [torch.cat([head, torch.randint(1, slots, (int(torch.randint(1, maxlen - shared + 1, (1,), generator=g)),),
                                                generator=g, dtype=torch.int32)]) for _ in range(n)]
        seq = torch.tensor([x.numel() for x in lists], dtype=torch.int32)
        return SimpleNamespace(is_prefill=False, n_rows=n, seq_lens=seq.to(dev), seq_lens_cpu=seq, kv_indptr=None,
                               kv_indices=torch.cat(lists).to(dev)), torch.cat(lists), seq

    def one():
        return be.forward_quant_fp8(q, 0) if quant else be.forward(q, None, None, 0, None, skip_store=True)

    be.prepare(batch(bs, 100)[0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        one()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = one()
    for n, shared in ((bs, 100), (17, 100), (5, 0), (bs, 0), (33, 40), (16, 0), (1, 64), (bs, 64)):
        print(f"graph of {bs} rows over {n}, {shared} shared", flush=True)
        b, kv, seq = batch(n, shared)
        be.prepare(b)
        graph.replay()
        torch.cuda.synchronize()
        start = torch.cumsum(seq, 0, dtype=torch.int32) - seq
        want = ops.paged_attention(q[:n].cpu(), k0, v0, kv, start, seq, SCALE).float().reshape(n, -1)
        if quant:
            got = out[0][:n].float().cpu() * out[1][:n].cpu()
            bound = 2.0 ** -4  # half an e4m3 step, and a bf16 one before it
        else:
            got, bound = out[:n].float().cpu().reshape(n, -1), 2.0 ** -7
        err = (got - want).abs().amax(1) / want.abs().amax(1)
        assert err.max().item() < bound, (n, shared, err.max().item())
    be.end_graph_decode()


@pytest.mark.parametrize("t", [40, 88])
def test_quant_into_given_buffers_allocates_nothing(dev, t):
    """With room for the codes, the scales and the bf16 rows, also where the keys are split (both sizes here)."""
    from flashrec_amd._lib import load
    from flashrec_amd.attention import attention_plan, paged_attention_quant_fp8

    q, k, v, idx, start, ln = _inputs(dev, 16, 8)
    plan = attention_plan(idx, start, ln, 16, 8)
    assert load().fr_paged_attention_waves(t, 16, 8, idx.numel()) > 1
    want = paged_attention_quant_fp8(q[:t], k, v, idx, start, ln, SCALE, group_prefix=plan)
    out, scale = torch.empty_like(want[0]), torch.empty_like(want[1])
    rows = torch.empty(t, 16, 128, dtype=torch.bfloat16, device=dev)
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    paged_attention_quant_fp8(q[:t], k, v, idx, start, ln, SCALE, group_prefix=plan, out=out, out_scale=scale, rows=rows)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
    assert torch.equal(out.view(torch.uint8), want[0].view(torch.uint8)) and torch.equal(scale, want[1])
    with pytest.raises(ValueError, match="rows"):
        paged_attention_quant_fp8(q[:t], k, v, idx, start, ln, SCALE, out=out, out_scale=scale, rows=rows[1:])
