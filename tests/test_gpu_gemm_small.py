"""The K-split GEMM of launches with few tiles (gemm_fp8_small.hip): integer
operands pin every output exactly on each of its tile shapes, for both weight
layouts, every epilogue and output type, partial tiles and K tails; outputs
past the last row and column stay untouched."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# the tile shapes by (rows x columns): 32x32, 32x64, 64x32, 64x64, 128x64, each
# whole, one short and one past its edges; K below one wave's share, one slot
# more than the waves', not a multiple of 128 or 256
SHAPES = [(1, 16, 16), (31, 48, 256), (32, 2048, 384), (33, 2048, 2048), (128, 2048, 1040),
          (1, 8224, 256), (20, 12288, 2048), (32, 16400, 272),
          (65, 4096, 640), (255, 2032, 2048), (64, 8192, 144),
          (129, 4096, 400), (511, 2048, 6144), (64, 12288, 512),
          (513, 2048, 4096), (1001, 2032, 4112), (1024, 2048, 6144)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_small_gemm_exact(dev, m, n, k):
    from flashrec_amd.kernel.sglops import (fp8_scaled_mm, fp8_scaled_mm_prearranged, fp8_scaled_mm_residual,
                                            fp8_scaled_mm_silu, prearrange_fp8_weight, silu_and_mul)

    print(f"small gemm {m}x{n}x{k}", flush=True)
    g = torch.Generator(device=dev).manual_seed(m + n + k)

    def ints(*shape):  # |sum| < 2^24 at every K here: fp32 adds exactly in any order
        return torch.randint(-3, 4, shape, generator=g, device=dev).float()

    a, w = ints(m, k), ints(n, k)
    sa = torch.exp2(torch.randint(-2, 3, (m, 1), generator=g, device=dev).float())
    sb = torch.exp2(torch.randint(-6, 0, (n,), generator=g, device=dev).float())
    ref = ((a.double() @ w.double().t()) * sa * sb).float()
    qa, qw = a.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn).t()
    pre = prearrange_fp8_weight(qw)
    bias = ints(n)
    res = ints(m, n)

    def guarded(cols, dt):
        buf = torch.full((m + 130, cols + 24), 7.0, dtype=dt, device=dev)
        return buf, buf[:m, :cols]

    def check(buf, got, want):
        assert torch.equal(got.float(), want.float())
        assert bool((buf[m:] == 7).all()) and bool((buf[:, want.shape[1]:] == 7).all())

    for dt in (torch.float32, torch.bfloat16, torch.float16):
        want = ref.to(dt)
        assert torch.equal(fp8_scaled_mm(qa, qw, sa, sb, dt), want)
        buf, out = guarded(n, dt)
        check(buf, fp8_scaled_mm_prearranged(qa, pre, sa, sb, dt, out=out), want)
        assert torch.equal(fp8_scaled_mm(qa, qw, sa, sb, dt, bias.to(dt)), (ref + bias).to(dt))
        if dt != torch.float32:
            want = (want.float() + res).to(dt)
            for call in (lambda r: fp8_scaled_mm_residual(qa, qw, sa, sb, r),
                         lambda r: fp8_scaled_mm_prearranged(qa, pre, sa, sb, residual=r)):
                buf, r = guarded(n, dt)
                r.copy_(res)
                check(buf, call(r), want)
    # gate/up chunks of 8: the same SiLU arithmetic as the row kernel's
    gu = ref.to(torch.bfloat16).view(m, n // 16, 2, 8)
    want = silu_and_mul(torch.cat([gu[:, :, 0].reshape(m, -1), gu[:, :, 1].reshape(m, -1)], 1))
    buf, out = guarded(n // 2, torch.bfloat16)
    check(buf, fp8_scaled_mm_silu(qa, qw, sa, sb, out=out), want)
    buf, out = guarded(n // 2, torch.bfloat16)
    check(buf, fp8_scaled_mm_prearranged(qa, pre, sa, sb, out=out, silu=True), want)


def test_small_gemm_layouts_agree(dev):
    """Random operands: both layouts add in one order, bit for bit, and the
    result is no further from float64 than an fp32 matmul's order allows."""
    from flashrec_amd.kernel.sglops import fp8_scaled_mm, fp8_scaled_mm_prearranged, prearrange_fp8_weight

    for m, n, k in ((20, 2048, 6144), (77, 4096, 2048), (400, 2048, 6144), (900, 2048, 6144)):
        g = torch.Generator(device=dev).manual_seed(m)
        a = torch.randn(m, k, generator=g, device=dev).to(torch.float8_e4m3fn)
        w = torch.randn(n, k, generator=g, device=dev).to(torch.float8_e4m3fn)
        one, onn = torch.ones(m, 1, device=dev), torch.ones(n, device=dev)
        got = fp8_scaled_mm_prearranged(a, prearrange_fp8_weight(w.t()), one, onn, torch.float32)
        assert torch.equal(got, fp8_scaled_mm(a, w.t(), one, onn, torch.float32)), (m, n, k)
        ref = a.double() @ w.double().t()
        bound = (a.double().abs() @ w.double().abs().t()) * (k * 2.0 ** -24)
        assert bool(((got.double() - ref).abs() <= bound).all()), (m, n, k)
