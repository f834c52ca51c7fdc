"""GEMM launches whose last row tile is partial: its rows take the staged
epilogue with the stores cut off at row M - 1.  Every variant gives the rows
of the same product over whole tiles bit for bit, and writes nothing past the
last row or column."""

import pytest
import torch

pytestmark = pytest.mark.gpu

GUARD = 7.0


def _guarded(m, n, dtype, dev):
    """[m, n] inside a buffer with guard rows below and guard columns beside it."""
    buf = torch.full((m + 300, n + 64), GUARD, dtype=dtype, device=dev)
    return buf, buf[:m, :n]


def _check(buf, got, want, m, n):
    assert torch.equal(got.float(), want[:m].float())
    assert bool((buf[m:] == GUARD).all()) and bool((buf[:, n:] == GUARD).all())


# one row, one short of a tile and odd counts in the last tile, for launches
# that take 256x256, 256x128 and 128x128 tiles
@pytest.mark.parametrize("m,n,k", [(1025, 12288, 256), (1279, 12288, 512), (4095, 2048, 256), (3073, 4096, 256),
                                   (1001, 2048, 384)])
def test_ragged_rows(dev, m, n, k):
    from flashrec_amd.kernel.sglops import (fp8_scaled_mm, fp8_scaled_mm_prearranged, fp8_scaled_mm_residual,
                                            fp8_scaled_mm_silu, prearrange_fp8_weight)

    print(f"ragged gemm {m}x{n}x{k}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + n)
    whole = (m + 255) // 256 * 256
    a = torch.randn(whole, k, generator=g, device=dev).to(torch.float8_e4m3fn)
    w = torch.randn(n, k, generator=g, device=dev).to(torch.float8_e4m3fn).t()
    sa = torch.rand(whole, 1, generator=g, device=dev) + 0.5
    sb = (torch.rand(n, generator=g, device=dev) + 0.5) * 0.05
    pre = prearrange_fp8_weight(w)
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        want = fp8_scaled_mm(a, w, sa, sb, dt)
        assert torch.equal(fp8_scaled_mm(a[:m], w, sa[:m], sb, dt).float(), want[:m].float()), dt
        buf, out = _guarded(m, n, dt, dev)
        _check(buf, fp8_scaled_mm_prearranged(a[:m], pre, sa[:m], sb, dt, out=out), want, m, n)
        if dt != torch.float32:
            res = torch.randn(whole, n, generator=g, device=dev).to(dt)
            want = (want.float() + res.float()).to(dt)
            for call in (lambda r: fp8_scaled_mm_residual(a[:m], w, sa[:m], sb, r),
                         lambda r: fp8_scaled_mm_prearranged(a[:m], pre, sa[:m], sb, residual=r)):
                buf, r = _guarded(m, n, dt, dev)
                r.copy_(res[:m])
                _check(buf, call(r), want, m, n)
    want = fp8_scaled_mm_silu(a, w, sa, sb)
    buf, out = _guarded(m, n // 2, torch.bfloat16, dev)
    _check(buf, fp8_scaled_mm_silu(a[:m], w, sa[:m], sb, out=out), want, m, n // 2)
    buf, out = _guarded(m, n // 2, torch.bfloat16, dev)
    _check(buf, fp8_scaled_mm_prearranged(a[:m], pre, sa[:m], sb, out=out, silu=True), want, m, n // 2)
