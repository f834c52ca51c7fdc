"""fp16 and fp32 rows: the workgroup-per-row kernel that aligned rows take and
the wave-per-row kernel that all others take give the same bits (rows of small
integers, whose sums of squares are exact in any order), with infinities, NaNs,
all-zero rows and widths at the edges of its 2048-element chunks."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("k", [8, 2040, 2048, 2056, 4096, 4104, 6144, 8192])
def test_aligned_rows_match_unaligned(dev, k, dtype):
    from flashrec_amd._lib import DTYPE_CODE, call

    print(f"rows {k} {dtype}", flush=True)
    m = 9
    g = torch.Generator(device=dev).manual_seed(k)

    def ints(*shape):
        return torch.randint(-9, 10, shape, generator=g, device=dev).to(dtype)

    x, u, res, w = ints(m, k), ints(m, k), ints(m, k), (1 + 0.25 * ints(k).abs())
    x[1] = 0
    x[2, k // 2] = float("inf")
    x[3, k - 1] = float("nan")
    gate = (x.float() / 2).to(dtype)
    code, st = DTYPE_CODE[dtype], torch.cuda.current_stream().cuda_stream

    def rows(t, pad):
        """t with row stride k + pad (pad 8: aligned, pad 1: not)."""
        buf = torch.zeros(m, t.shape[1] + pad, dtype=dtype, device=dev)
        buf[:, : t.shape[1]] = t
        return buf

    def run(pad):
        out = {}
        q = torch.zeros(m, k, dtype=torch.uint8, device=dev)
        s = torch.zeros(m, device=dev)
        xs, gu = rows(x, pad), rows(torch.cat([gate, u], 1), pad)

        def quantised(name, fn, *args):
            call(fn, *args, q.data_ptr(), s.data_ptr(), st)
            out[name] = (q.clone(), s.view(torch.int32).clone())

        quantised("quant", "fr_per_token_quant_fp8", xs.data_ptr(), code, m, k, k + pad)
        quantised("rms", "fr_rms_quant_fp8", xs.data_ptr(), code, k + pad, None, 0, w.data_ptr(), m, k, 1e-6)
        r = rows(res, pad)
        quantised("add", "fr_rms_quant_fp8", xs.data_ptr(), code, k + pad, r.data_ptr(), k + pad, w.data_ptr(), m, k,
                  1e-6)
        out["residual"] = (r[:, :k].clone(),)
        assert bool((r[:, k:] == 0).all())
        quantised("silu", "fr_silu_quant_fp8", gu.data_ptr(), code, 2 * k + pad, m, k)
        y = torch.full((m, k + pad), 7.0, dtype=dtype, device=dev)
        call("fr_rmsnorm", xs.data_ptr(), code, k + pad, None, 0, w.data_ptr(), y.data_ptr(), k + pad, m, k, 1e-6, st)
        out["rmsnorm"] = (y[:, :k].clone(),)
        assert bool((y[:, k:] == 7).all())
        y = torch.full((m, k + pad), 7.0, dtype=dtype, device=dev)
        call("fr_silu_and_mul", gu.data_ptr(), code, 2 * k + pad, y.data_ptr(), k + pad, m, k, st)
        out["mul"] = (y[:, :k].clone(),)
        assert bool((y[:, k:] == 7).all())
        return out

    aligned, other = run(8), run(1)
    for name in aligned:
        for a, b in zip(aligned[name], other[name]):
            if a.is_floating_point():
                a, b = a.float(), b.float()
                assert bool(((a == b) | (a.isnan() & b.isnan())).all()), name
            elif a.dtype == torch.uint8:  # a NaN code's sign is not pinned
                nan = ((a & 0x7F) == 0x7F) & ((b & 0x7F) == 0x7F)
                assert bool(((a == b) | nan).all()), name
            else:  # scales, as bits; NaN payloads are not pinned
                fa, fb = a.view(torch.float32), b.view(torch.float32)
                assert bool(((a == b) | (fa.isnan() & fb.isnan())).all()), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("k", [64, 504, 512, 520, 1016, 1024, 1032])
def test_narrow_rows_match_unaligned(dev, k, dtype):
    """The same at the edges of the widths that take a wave per row (9 rows: two
    workgroups of four and one of one)."""
    test_aligned_rows_match_unaligned(dev, k, dtype)


def test_more_rows_than_workgroups(dev):
    """Past 2^24 rows: a workgroup of 256 threads for each would be more than a
    launch holds."""
    from flashrec_amd.kernel.sglops import per_token_quant_fp8

    m = (1 << 24) + 5
    x = torch.zeros(m, 8, dtype=torch.float16, device=dev)
    x[-3:] = torch.arange(8, device=dev)
    q, s = per_token_quant_fp8(x)
    want = torch.full((m,), 1e-12, device=dev)
    want[-3:] = 7.0
    assert torch.equal(s.view(-1), want / 448)
    assert bool((q[:-3].view(torch.uint8) == 0).all()) and torch.equal(
        q[-1].float(), (torch.arange(8, device=dev) / s[-1]).to(torch.float8_e4m3fn).float())
