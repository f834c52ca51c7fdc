"""The top-k's bins: rows of both signs, of one value, of a few subnormals, with
one far outlier, with masked entries (-1e9, the lowest float, -inf), with signed
zeros, each against a stable sort, for whole rows (binned by score) and ragged
ones (binned by the key's bits)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(kind, v, g):
    x = torch.randn(6, v, generator=g) * 0.9
    if kind == "one":
        return torch.full((6, v), -1.25)
    if kind == "subnormal":
        return torch.randint(0, 5, (6, v), generator=g).float() * 1.4e-45
    if kind == "outlier":
        x[:, 3] = 60.0
        x[1:3, 4] = 1e6
    if kind == "masked":
        keep = torch.rand(6, v, generator=g) < 0.4
        low = torch.tensor([-1e9, -3.4028235e38, float("-inf")]).repeat(2)[:, None]
        x = torch.where(keep, x, low)
    if kind == "zeros":
        x = x.round() * torch.where(torch.rand(6, v, generator=g) < 0.5, -1.0, 1.0)
    if kind == "negative":
        x = torch.log_softmax(x, -1)
    return x


@pytest.mark.parametrize("kind", ["both", "one", "subnormal", "outlier", "masked", "zeros", "negative"])
@pytest.mark.parametrize("v,c", [(8192, 1024), (4096, 100), (1024, 1024), (8190, 1000)])
def test_row_topk_bins(dev, v, c, kind):
    from flashrec_amd.kernel.beam_trie import row_topk
    from flashrec_amd.kernel.sglops import log_softmax_f32

    print(f"top-k bins {kind} {v} -> {c}", flush=True)
    x = _rows(kind, v, torch.Generator().manual_seed(v + c)).to(torch.float32)

    def check(got, scores):
        vals, idx = torch.sort(scores, dim=-1, descending=True, stable=True)
        assert torch.equal(got[0].cpu(), vals[:, :c]) and torch.equal(got[1].cpu(), idx[:, :c])
        assert torch.equal(got[0].cpu().view(torch.int32), torch.gather(scores, 1, idx[:, :c]).view(torch.int32))

    check(row_topk(x.to(dev), c), x)
    if kind != "masked":  # (a row's log-probabilities as the log-softmax kernel writes them)
        check(row_topk(x.to(dev), c, log_softmax=True), log_softmax_f32(x.to(dev)).cpu())


@pytest.mark.parametrize("kind", ["both", "one", "outlier", "masked", "zeros"])
@pytest.mark.parametrize("v,c", [(16384, 1024), (16384, 40), (2048, 700)])
def test_row_topk_bins_widest(dev, v, c, kind):
    """64 keys a thread (two words of boundary-bin bits) and 8."""
    test_row_topk_bins(dev, v, c, kind)
