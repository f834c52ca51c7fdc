"""The beam step's selection (histogram select, bin sort, allow rows through
LDS) at the shapes where it can go wrong: crowded bins and scores that all tie,
infinities with masking off, K at the edges of its sorts and caps, allow rows of
16-byte multiples up to and past the LDS row, one candidate more than kept."""

import pytest
import torch

from test_gpu_beam import _case, _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bw,c,k,vocab", [(2, 1, 1, 1, 16), (1, 16, 64, 64, 1024), (1, 33, 40, 65, 1040),
                                            (2, 64, 64, 512, 768), (1, 130, 16, 513, 1008), (1, 512, 4, 1023, 32),
                                            (3, 512, 64, 1024, 768)])
def test_select_shapes(dev, n, bw, c, k, vocab):
    print(f"select {n}x{bw}x{c} top {k} of {vocab}", flush=True)
    _compare(dev, _case(n, bw, c, vocab, 20, 0.8, 11 * bw + k), k)


@pytest.mark.parametrize("k", [7, 64, 200, 512])
def test_crowded_scores(dev, k):
    """All scores equal; all but a few equal and the rest far away; scores a
    few ulps apart around one far outlier."""
    args = list(_case(2, 64, 32, 256, 20, 0.9, k))
    cum, lp = args[0], args[1]
    for fill in (lambda s: torch.zeros_like(s), lambda s: torch.where(s > 1.5, 1e30, 0.0).to(s.dtype),
                 lambda s: (1.0 + (s * 8).floor() * 2.0 ** -23) - 1e20 * (s > 2.5)):
        args[0] = torch.zeros_like(cum)
        args[1] = torch.sort(fill(lp), dim=-1, descending=True).values
        _compare(dev, tuple(args), k)


def test_infinite_scores_unmasked(dev):
    args = list(_case(1, 48, 32, 256, 20, 0.9, 5))
    lp = args[1].clone()
    lp[0, ::5, :] = float("-inf")
    lp[0, 3, :2] = float("inf")
    args[1] = torch.sort(lp, dim=-1, descending=True).values
    _compare(dev, tuple(args), 48, apply_mask=False)
    _compare(dev, tuple(args), 48)


@pytest.mark.parametrize("n,bw,c,k", [(2, 3, 64, 2), (1, 17, 65, 32), (1, 20, 256, 33), (2, 20, 257, 63), (1, 16, 1024, 1024),
                                      (1, 17, 64, 512), (1, 32, 40, 513), (1, 1030, 1, 1), (3, 1100, 2, 17)])
def test_narrow_beams_and_few_lists(dev, n, bw, c, k):
    """Candidates a beam around one and four chunks of 64, slices' lists around
    1024 keys in all (17 and 32 beams are two slices), more lists than a group."""
    print(f"narrow {n}x{bw}x{c} top {k}", flush=True)
    _compare(dev, _case(n, bw, c, 768, 20, 0.8, 13 * bw + c), k)
