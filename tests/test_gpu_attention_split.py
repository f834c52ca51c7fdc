"""Paged attention over segments and key splits: prompts that meet inside a
query group, beams of several requests in one group, shared prefixes that are
no multiple of 32, single tokens, empty lists, and the keys of an item split
over 1, 2, 4 and 8 waves, each against the fp32 oracle."""

import pytest
import torch

from oracle import ops

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn
SCALE = 128 ** -0.5


def _case(kind, seed):
    """(slot lists, one per token; tokens that read the same list share it)."""
    g = torch.Generator().manual_seed(seed)
    perm = (1 + torch.randperm(4000, generator=g)).to(torch.int32)

    def fresh(n, at=[0]):
        at[0] = (at[0] + n) % 3000
        return perm[at[0]:at[0] + n]

    rows = []  # (list, length seen)
    if kind == "prompts":  # causal prompts of odd lengths, one with a cached prefix, one of a single token
        for cached, n in ((0, 45), (70, 9), (0, 1), (0, 33), (5, 100)):
            lst = fresh(cached + n)
            rows += [(lst, cached + j + 1) for j in range(n)]
    elif kind == "beams":  # requests of odd beam counts, prefixes around the blocks, own slots past them
        for prefix, beams, own in ((200, 21, 2), (31, 9, 3), (33, 18, 1), (64, 7, 40), (95, 5, 0)):
            head = fresh(prefix)
            for _ in range(beams):
                lst = torch.cat([head, fresh(own)]) if own else head.clone()
                rows.append((lst, prefix + own))
    else:  # unrelated rows, empty ones among them
        for n in (0, 1, 31, 32, 33, 0, 64, 257, 7, 96, 1, 130, 5, 40, 41, 42, 43, 300):
            rows.append((fresh(n), n))
    idx, start, lens, seen = [], [], [], {}
    for lst, n in rows:
        if id(lst) not in seen:
            seen[id(lst)] = sum(int(x.numel()) for x in idx)
            idx.append(lst)
        start.append(seen[id(lst)])
        lens.append(n)
    return torch.cat(idx), torch.tensor(start, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)


def _run(dev, q, k, v, idx, start, lens, waves, plan):
    from flashrec_amd._lib import call
    from flashrec_amd.attention import attention_plan

    d = [x.to(dev) for x in (q, k, v, idx, start, lens)]
    t, hq, hk = q.shape[0], q.shape[1], k.shape[1]
    gp = attention_plan(d[3], d[4], d[5], hq, hk) if plan else None
    buf = torch.full((t + 2, hq, 128), 7.0, dtype=torch.bfloat16, device=dev)
    call("fr_paged_attention_split_fp8", d[0].data_ptr(), hq * 128, 128, d[1].data_ptr(), hk * 128, 128,
         d[2].data_ptr(), hk * 128, 128, k.shape[0], d[3].data_ptr(), d[4].data_ptr(), d[5].data_ptr(),
         buf.data_ptr(), hq * 128, 128, t, hq, hk, 128, SCALE, 0 if gp is None else gp.data_ptr(), waves,
         torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert bool((buf[t:] == 7).all())
    return buf[:t].cpu()


@pytest.mark.parametrize("hq,hk", [(16, 8), (8, 8), (16, 4), (16, 2)])
@pytest.mark.parametrize("kind", ["prompts", "beams", "rows"])
def test_segments_and_splits(dev, kind, hq, hk):
    print(f"attention {kind} {hq}/{hk}", flush=True)
    idx, start, lens = _case(kind, 3)
    g = torch.Generator().manual_seed(5)
    k = torch.randn(4001, hk, 128, generator=g).to(E4M3)
    v = torch.randn(4001, hk, 128, generator=g).to(E4M3)
    q = (2 * torch.randn(lens.numel(), hq, 128, generator=g)).to(torch.bfloat16)
    want = ops.paged_attention(q, k, v, idx, start, lens, SCALE).float()
    whole = _run(dev, q, k, v, idx, start, lens, 1, False)
    for waves in (1, 2, 4, 8):
        for plan in (False, True):
            got = _run(dev, q, k, v, idx, start, lens, waves, plan)
            if waves == 1:
                assert torch.equal(got, whole)
            # a probability rounded to bf16 (2^-9 of it) moves a row by at most
            # 2^-9 max |v| (|v| < 5), the output's own rounding by 2^-9 of it
            err = (got.float() - want).abs().max().item()
            assert err < 2.0 ** -9 * 5 + 2.0 ** -8 * want.abs().max().item(), (waves, plan, err)


@pytest.mark.parametrize("waves", [1, 4])
def test_nan_stays_with_its_readers(dev, waves):
    """A NaN V row inside a prompt's first tokens reaches the tokens that see it
    and no other, also where tokens of two prompts meet in one group."""
    idx, start, lens = _case("prompts", 4)
    g = torch.Generator().manual_seed(6)
    k = torch.randn(4001, 8, 128, generator=g).to(E4M3)
    v = torch.randn(4001, 8, 128, generator=g).to(E4M3)
    q = torch.randn(lens.numel(), 16, 128, generator=g).to(torch.bfloat16)
    slot = int(idx[7])  # position 7 of the first prompt
    clean = _run(dev, q, k, v, idx, start, lens, waves, True)
    v.view(torch.uint8)[slot] = 0x7F
    got = _run(dev, q, k, v, idx, start, lens, waves, True)
    sees = torch.zeros(lens.numel(), dtype=torch.bool)
    for t in range(lens.numel()):
        sees[t] = slot in idx[start[t]:start[t] + lens[t]].tolist()
    assert bool(torch.isnan(got[sees].float()).all())
    few = ~sees & (start == start[0]) & (lens < 16)  # the group before the first whole one
    assert int(few.sum()) == 7 and bool(torch.isfinite(got[~sees].float()).all())
    assert (got[few].float() - clean[few].float()).abs().max().item() < 2.0 ** -7 * 5


def test_wave_rule():
    """Whole launches stay unsplit, few items and prompts are split; an unknown head ratio or no tokens: 1."""
    from flashrec_amd._lib import load

    w = load().fr_paged_attention_waves
    assert w(4096, 16, 8, 4096 * 131) == 1 and w(0, 16, 8, 0) == 1 and w(10, 15, 4, 10) == 1
    assert w(50, 16, 8, 50 * 202) > 1 and w(1999, 16, 8, 1999) > 1


@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("hq,hk", [(16, 8), (8, 8), (16, 4), (16, 2)])
def test_probabilities_keep_32_bits(dev, hq, hk, waves):
    """Tokens with lists of their own: the difference of two nearly equal
    probabilities, times 448.  It is 2^-11 of them and more, so an error of
    2^-17 in each, which 16 bits leave, is up to 2^-5 of the result, where
    32-bit scores, powers and sums leave about 2^-10; the output rounds by 2^-8."""
    print(f"probabilities {hq}/{hk}, {waves} waves", flush=True)
    t = 70
    g = torch.Generator().manual_seed(11)
    k = torch.zeros(4, hk, 128)
    k[1:3, :, 0] = torch.tensor([1.0, 1.125])[:, None]
    k[3, :, 1] = 1.0
    v = torch.tensor([0.0, 448.0, -448.0, 0.0])[:, None, None].expand(4, hk, 128).contiguous()
    q = torch.zeros(t, hq, 128)
    q[:, :, 0] = 0.05 + 0.15 * torch.rand(t, hq, generator=g)
    q[:, :, 1] = 8 * torch.randn(t, hq, generator=g)
    q = q.to(torch.bfloat16)
    idx = torch.tensor([1, 2, 3], dtype=torch.int32).repeat(t)
    start, lens = torch.arange(t, dtype=torch.int32) * 3, torch.full((t,), 3, dtype=torch.int32)
    got = _run(dev, q, k.to(E4M3), v.to(E4M3), idx, start, lens, waves, True).double()
    a, c = q[..., 0].double(), q[..., 1].double()
    p = torch.softmax(torch.stack([a, 1.125 * a, c], -1) * SCALE, -1)
    want = ((p[..., 0] - p[..., 1]) * 448)[..., None]
    err = ((got - want) / want).abs().max().item()
    assert err < 2.0 ** -8 + 2.0 ** -9, err


@pytest.mark.parametrize("waves", [1, 2, 4])
def test_nan_in_a_group_of_two_prompts(dev, waves):
    """The same where the segments of a group go to the waves in turn (two and
    more, on two waves): tokens 32 .. 44 of the first prompt share a group with
    the second one's first; its position 40 is NaN."""
    idx, start, lens = _case("prompts", 4)
    g = torch.Generator().manual_seed(8)
    k = torch.randn(4001, 8, 128, generator=g).to(E4M3)
    v = torch.randn(4001, 8, 128, generator=g).to(E4M3)
    q = torch.randn(lens.numel(), 16, 128, generator=g).to(torch.bfloat16)
    clean = _run(dev, q, k, v, idx, start, lens, waves, True)
    v.view(torch.uint8)[int(idx[40])] = 0x7F
    got = _run(dev, q, k, v, idx, start, lens, waves, True)
    sees = (start == start[0]) & (lens > 40)
    assert int(sees.sum()) == 5 and bool(torch.isnan(got[sees].float()).all())
    assert bool(torch.isfinite(got[~sees].float()).all())
    assert (got[~sees].float() - clean[~sees].float()).abs().max().item() < 2.0 ** -7 * 5
