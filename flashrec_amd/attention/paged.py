"""Paged fp8 attention backend, interface of ``flashrec.attention.flashinfer``.

Reference: python/flashrec/attention/flashinfer.py:73-431 (``AttentionBackend``).
The reference plans FlashInfer wrappers per batch and runs them per layer; the
result it defines is that of its ``_sdpa`` fallback (:380-431).  Here the plan
is two int32 arrays per query token — where its slot list starts in
``kv_indices`` and how many slots it sees — and every layer runs the gfx950
kernel ``fr_paged_attention_fp8`` over the e4m3 pool.  The plan is built in
``prepare`` (outside graph capture, as the reference's is); under graph decode
it is written into persistent per-batch-size buffers, so ``forward`` allocates
only its output and can be captured.
"""

from __future__ import annotations

from functools import lru_cache
from typing import Dict, List, Optional, Tuple

import torch

from flashrec_amd._lib import DTYPE_CODE, Unsupported, call, load, require_device, stream_of


class AttentionBackend:
    """Drop-in for the reference backend (flashinfer.py:73-141): same
    constructor, ``prepare`` / ``forward`` and graph-decode hooks."""

    def __init__(
        self,
        kv_pool,
        num_qo_heads: int,
        num_kv_heads: int,
        head_dim: int,
        backend: str = "hip",
        fi_backend: str = "fa2",
    ):
        if num_qo_heads % num_kv_heads != 0:
            raise ValueError("num_qo_heads must be a multiple of num_kv_heads")
        if head_dim != 128:
            raise ValueError("the paged attention kernel takes head_dim 128")
        self.kv_pool = kv_pool
        self.num_qo_heads = int(num_qo_heads)
        self.num_kv_heads = int(num_kv_heads)
        self.head_dim = int(head_dim)
        self.n_rep = self.num_qo_heads // self.num_kv_heads
        self.device = kv_pool.device
        self.backend = backend
        self.fi_backend = fi_backend
        self.q_dtype = torch.bfloat16
        # the reference shares one workspace between prefill and decode when it
        # cannot allocate two; this backend has no workspace to overlap
        self.prefill_overlap_ok = True
        self.scale = self.head_dim ** -0.5
        self._plan: Optional[Dict[str, torch.Tensor]] = None
        self._graph_bufs: Dict[int, Dict[str, torch.Tensor]] = {}
        self._graph_bs: Optional[int] = None

    # ---------------------------------------------------------- graph decode
    def init_graph_wrappers(self, capture_bs: List[int], max_seq_len: int) -> None:
        """Persistent plan buffers per captured batch size (flashinfer.py:143-185)."""
        max_seq_len = max(int(max_seq_len), 1)
        for bs in capture_bs:
            bs = int(bs)
            if bs <= 0 or bs in self._graph_bufs:
                continue
            dev = self.device
            self._graph_bufs[bs] = {
                "indptr": torch.zeros(bs + 1, dtype=torch.int32, device=dev),
                "indices": torch.zeros(bs * max_seq_len, dtype=torch.int32, device=dev),
                "last": torch.ones(bs, dtype=torch.int32, device=dev),
                "kv_len": torch.zeros(bs, dtype=torch.int32, device=dev),
                "group_prefix": _plan_rows(
                    torch.zeros(plan_size(bs, self.num_qo_heads, self.num_kv_heads), dtype=torch.int32, device=dev),
                    bs, self.num_qo_heads, self.num_kv_heads),
            }

    def graph_bufs(self, bs: int) -> Optional[dict]:
        return self._graph_bufs.get(int(bs))

    def begin_graph_decode(self, bs: int) -> None:
        if int(bs) not in self._graph_bufs:
            raise RuntimeError(f"no graph plan buffers for bs={bs}")
        self._graph_bs = int(bs)

    def end_graph_decode(self) -> None:
        self._graph_bs = None

    # ----------------------------------------------------------------- plan
    def prepare(self, batch) -> None:
        """Per-token slot ranges for every layer of this batch (flashinfer.py:201-210),
        and the shared-prefix plan of its query groups (one kernel, reused by
        every layer's attention)."""
        if batch.kv_indices is None:
            self._plan = None
            return
        if batch.is_prefill:
            self._plan = self._plan_prefill(batch)
        else:
            self._plan = self._plan_decode(batch)
        n = int(self._plan["start"].numel())
        bufs = self._graph_bufs.get(self._graph_bs) if self._graph_bs is not None else None
        gp = None
        if bufs is not None and not batch.is_prefill:
            gp = bufs["group_prefix"]
        self._plan["group_prefix"] = attention_plan(self._plan["indices"], self._plan["start"],
                                                    self._plan["len"], self.num_qo_heads,
                                                    self.num_kv_heads, out=gp)

    def _plan_decode(self, batch) -> Dict[str, torch.Tensor]:
        n = int(batch.n_rows)
        seq = batch.seq_lens.view(-1)[:n].to(device=self.device, dtype=torch.int32)
        kv = batch.kv_indices.view(-1)
        if kv.dtype != torch.int32:
            kv = kv.to(dtype=torch.int32)
        bufs = self._graph_bufs.get(self._graph_bs) if self._graph_bs is not None else None
        if bufs is not None:
            # indptr[0] stays 0 (zeros at creation); the cumsum fills [1:]
            torch.cumsum(seq, dim=0, out=bufs["indptr"][1 : n + 1])
            bufs["kv_len"][:n].copy_(seq)
            nidx = int(kv.numel())
            if nidx > 0 and kv.data_ptr() != bufs["indices"].data_ptr():
                bufs["indices"][:nidx].copy_(kv, non_blocking=True)
            # (no "entries": a captured launch serves every length its buffers
            # hold, so its split is chosen for their capacity.  us, 16/8 heads:
            # 2048 x 130 in rows of 4096 slots 21.5 for 19.6 unsplit, where 1248 x
            # 1133 unsplit would take 180 for 73)
            return {"indices": bufs["indices"], "start": bufs["indptr"][:n], "len": bufs["kv_len"][:n]}
        indptr = batch.kv_indptr
        if indptr is None:
            indptr = torch.zeros(n + 1, dtype=torch.int32, device=self.device)
            torch.cumsum(seq, dim=0, out=indptr[1:])
        indptr = indptr.view(-1).to(device=self.device, dtype=torch.int32)
        return {"indices": kv.contiguous(), "start": indptr[:n].contiguous(), "len": seq.contiguous()}

    def _plan_prefill(self, batch) -> Dict[str, torch.Tensor]:
        """Causal prefill (flashinfer.py:351-378, :409-422): token j of a row with
        prefix P sees the row's first P + j + 1 slots."""
        n = int(batch.n_rows)
        seq = [int(x) for x in batch.seq_lens_cpu.view(-1)[:n].tolist()]
        ext = [int(e) for e in (batch.extend_seq_lens or [1] * n)]
        prefix = batch.extend_prefix_lens or [s - e for s, e in zip(seq, ext)]
        start: List[int] = []
        length: List[int] = []
        off = 0
        for i in range(n):
            for j in range(ext[i]):
                start.append(off)
                length.append(int(prefix[i]) + j + 1)
            off += seq[i]
        kv = batch.kv_indices.view(-1).to(device=self.device, dtype=torch.int32).contiguous()
        # for the split of the keys over waves: tokens that share their prompt's
        # list count one slot each (so that a long cached prefix is not taken for
        # lists of their own), else each reads its own
        shared = len(start) >= 8 * n
        return {
            "indices": kv,
            "entries": len(start) if shared else sum(length),
            "start": torch.tensor(start, dtype=torch.int32).to(self.device),
            "len": torch.tensor(length, dtype=torch.int32).to(self.device),
        }

    # ------------------------------------------------------------------ run
    @torch.compiler.disable
    def forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer_id: int, batch,
                skip_store: bool = False) -> torch.Tensor:
        """q/k/v: [T, H, D] (k/v kv-heads).  Writes the new KV, then attends
        (flashinfer.py:212-238).  Returns [T, Hq, D] bf16."""
        if not skip_store:
            self.kv_pool.store(layer_id, k, v, batch.out_cache_loc)
        if self._plan is None:
            raise RuntimeError("AttentionBackend.forward before prepare() (kv_indices required)")
        return paged_attention(q, self.kv_pool.k_cache(layer_id), self.kv_pool.v_cache(layer_id),
                               self._plan["indices"], self._plan["start"], self._plan["len"],
                               self.scale, group_prefix=self._plan.get("group_prefix"),
                               entries=self._plan.get("entries"))


    @torch.compiler.disable
    def forward_quant_fp8(self, q: torch.Tensor, layer_id: int) -> Tuple[torch.Tensor, torch.Tensor]:
        """Attention over the stored KV fused with the o projection's per-token
        e4m3 quant: (codes [T, Hq * D], scales [T, 1]).  The new KV must be
        stored already (the fused QK-norm/RoPE/KV write does it)."""
        if self._plan is None:
            raise RuntimeError("AttentionBackend.forward_quant_fp8 before prepare() (kv_indices required)")
        return paged_attention_quant_fp8(q, self.kv_pool.k_cache(layer_id), self.kv_pool.v_cache(layer_id),
                                         self._plan["indices"], self._plan["start"], self._plan["len"],
                                         self.scale, group_prefix=self._plan.get("group_prefix"),
                                         entries=self._plan.get("entries"))


def plan_size(T: int, hq: int, hk: int) -> int:
    """Entries of an attention plan's buffer for T query tokens: one record per
    group of 32 / (hq / hk) of them."""
    n = int(load().fr_paged_attention_plan_size(int(T), int(hq), int(hk)))
    if n < 0:
        raise ValueError(f"unsupported head ratio {hq}/{hk}")
    return n


@lru_cache(maxsize=64)
def _record_size(hq: int, hk: int) -> int:
    return plan_size(1, hq, hk)


def _groups(T: int, hq: int, hk: int) -> Tuple[int, int]:
    """(query groups of T tokens, entries of a group's record)."""
    stride = _record_size(int(hq), int(hk))
    return -(-int(T) * (int(hq) // int(hk)) // 32), stride


def _plan_rows(buf: torch.Tensor, T: int, hq: int, hk: int) -> torch.Tensor:
    """The records at the front of a flat plan buffer as attention_plan returns
    them: a strided view with one entry, its shared prefix, per group."""
    groups, stride = _groups(T, hq, hk)
    return buf.reshape(-1)[: groups * stride].view(groups, stride)[:, 0]


def _plan_records(plan: torch.Tensor, groups: int, stride: int) -> bool:
    """Whether ``plan`` (a view as _plan_rows makes it, or a flat buffer) has
    room for the whole records of ``groups`` groups."""
    if plan.dim() == 1 and plan.numel() >= groups and plan.stride(0) == stride:
        return plan.storage_offset() + groups * stride <= plan.untyped_storage().nbytes() // 4
    return plan.is_contiguous() and plan.numel() >= groups * stride


def _check_plan_buffer(plan: torch.Tensor, groups: int, records: bool) -> None:
    if plan.dtype != torch.int32 or not (records or plan.is_contiguous()) or plan.numel() < groups:
        raise ValueError(f"a plan is what attention_plan returns for the same slot lists, at least {groups} groups "
                         "of them, or a contiguous int32 tensor of as many entries")
    require_device(plan)


def attention_plan(kv_indices: torch.Tensor, kv_start: torch.Tensor, kv_len: torch.Tensor,
                   hq: int, hk: int, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The shared slot prefix (rounded down to 32) of each group of 32 / (hq /
    hk) consecutive query tokens: computed once per batch, passed to every
    layer's ``paged_attention`` as ``group_prefix``.  What is returned is a
    strided view of one record per group, which holds the kernels' own entries
    too (how the group's tokens fall into runs with common keys); ``out`` may
    be such a view, a flat buffer of ``plan_size`` entries, which it then views,
    or a contiguous tensor of one entry per group, which receives the prefixes
    alone."""
    require_device(kv_indices, kv_start, kv_len)
    T = int(kv_start.numel())
    groups, stride = _groups(T, hq, hk)
    if out is None:
        plan = rows = torch.empty((max(groups, 1), stride), dtype=torch.int32, device=kv_start.device).select(1, 0)
    else:
        records = _plan_records(out, groups, stride)
        _check_plan_buffer(out, groups, records)
        plan = out if records else torch.empty(groups * stride, dtype=torch.int32, device=kv_start.device)
        rows = out if out.dim() == 1 and out.stride(0) == stride else _plan_rows(plan, T, hq, hk)
    call("fr_paged_attention_plan", kv_indices.data_ptr(), kv_start.data_ptr(), kv_len.data_ptr(),
         T, int(hq), int(hk), plan.data_ptr(), stream_of(kv_start))
    if out is not None and plan is not out:
        out.view(-1)[:groups].copy_(rows)
        return out
    return rows


def _check_plan(group_prefix: Optional[torch.Tensor], T: int, hq: int, hk: int) -> int:
    """The device pointer of the plan's records after checking that it holds
    those the kernels read for T tokens; 0, and each call finds the shared
    prefixes itself, without a plan and for one of bare prefixes."""
    if group_prefix is None:
        return 0
    groups, stride = _groups(T, hq, hk)
    records = _plan_records(group_prefix, groups, stride)
    _check_plan_buffer(group_prefix, groups, records)
    return group_prefix.data_ptr() if records else 0


def _waves(T: int, hq: int, hk: int, kv_indices: torch.Tensor, entries: Optional[int]) -> int:
    return int(load().fr_paged_attention_waves(T, hq, hk, kv_indices.numel() if entries is None else int(entries)))


def _check_attention_inputs(q, k_cache, v_cache, kv_indices, kv_start, kv_len):
    require_device(q, k_cache, v_cache, kv_indices, kv_start, kv_len)
    if q.dtype != torch.bfloat16:
        raise TypeError("paged_attention takes bf16 queries")
    if k_cache.dtype != torch.float8_e4m3fn or v_cache.dtype != torch.float8_e4m3fn:
        raise TypeError("paged_attention reads an e4m3 KV pool")
    for t in (kv_indices, kv_start, kv_len):
        if t.dtype is not torch.int32 or not t.is_contiguous():
            raise TypeError("kv_indices / kv_start / kv_len must be contiguous int32")
    T, Hq, D = q.shape
    slots, Hk, Dk = k_cache.shape
    if Dk != D or v_cache.shape != k_cache.shape or q.stride(2) != 1:
        raise ValueError("q / cache shapes disagree")
    if k_cache.stride(2) != 1 or v_cache.stride(2) != 1:
        raise ValueError("caches need a unit inner stride")
    if kv_start.numel() < T or kv_len.numel() < T:
        raise ValueError("one kv_start / kv_len entry per query token")
    return T, Hq, D, slots, Hk


def paged_attention_quant_fp8(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                              kv_indices: torch.Tensor, kv_start: torch.Tensor, kv_len: torch.Tensor,
                              scale: float, group_prefix: Optional[torch.Tensor] = None,
                              out: Optional[torch.Tensor] = None, out_scale: Optional[torch.Tensor] = None,
                              entries: Optional[int] = None, rows: Optional[torch.Tensor] = None
                              ) -> Tuple[torch.Tensor, torch.Tensor]:
    """``per_token_quant_fp8(paged_attention(...).reshape(T, -1))`` in one
    kernel: the o projection's e4m3 input ``[T, Hq * D]`` and its scales
    ``[T, 1]`` (qwen3.py:131-134 -> linear.py:118-151), bit-for-bit the two
    steps' result.  Head layouts the fused kernel does not take (more than 8
    kv heads, 8 query heads per kv head), and launches with too few query
    groups to fill the chip, run the two steps; the attention's bf16 rows then go
    to ``rows`` (contiguous, [T, Hq, D]) or, without it, to a tensor allocated
    here, as do codes for an ``out`` with gaps between its rows.  With ``rows``,
    ``out_scale`` and a contiguous ``out`` given nothing is allocated."""
    T, Hq, D, slots, Hk = _check_attention_inputs(q, k_cache, v_cache, kv_indices, kv_start, kv_len)
    if out is None:
        out = torch.empty(T, Hq * D, dtype=torch.float8_e4m3fn, device=q.device)
    if out_scale is None:
        out_scale = torch.empty(T, 1, dtype=torch.float32, device=q.device)
    if (out.dtype != torch.float8_e4m3fn or out.dim() != 2 or out.shape[0] != T or out.shape[1] != Hq * D
            or out.stride(1) != 1):
        raise ValueError("out must be [T, Hq * D] float8_e4m3fn with a unit inner stride")
    if out_scale.dtype != torch.float32 or out_scale.numel() != T or not out_scale.is_contiguous():
        raise ValueError("out_scale must hold T contiguous fp32 values")
    if rows is not None and (rows.dtype != torch.bfloat16 or tuple(rows.shape) != (T, Hq, D)
                             or not rows.is_contiguous()):
        raise ValueError("rows must be contiguous [T, Hq, D] bf16")
    require_device(out, out_scale, rows)
    # where paged_attention splits its items' keys over waves, the quant runs
    # on its rows (one more launch of 3 us; 512 rows over 1503 keys take 89 us
    # fused and unsplit, 25 us so)
    waves = _waves(T, Hq, Hk, kv_indices, entries)
    plan = _check_plan(group_prefix, T, Hq, Hk)
    if waves == 1:
        try:
            call("fr_paged_attention_quant_fp8",
                 q.data_ptr(), q.stride(0), q.stride(1),
                 k_cache.data_ptr(), k_cache.stride(0), k_cache.stride(1),
                 v_cache.data_ptr(), v_cache.stride(0), v_cache.stride(1),
                 slots, kv_indices.data_ptr(), kv_start.data_ptr(), kv_len.data_ptr(),
                 out.data_ptr(), out.stride(0), out_scale.data_ptr(),
                 T, Hq, Hk, D, float(scale), plan, stream_of(q))
            return out, out_scale
        except Unsupported:
            pass
    o = torch.empty(T, Hq, D, dtype=torch.bfloat16, device=q.device) if rows is None else rows
    _attend(q, k_cache, v_cache, kv_indices, kv_start, kv_len, scale, o, plan, waves)
    codes = out if out.is_contiguous() else torch.empty((T, Hq * D), dtype=out.dtype, device=out.device)
    call("fr_per_token_quant_fp8", o.data_ptr(), DTYPE_CODE[o.dtype], T, Hq * D, Hq * D, codes.data_ptr(),
         out_scale.data_ptr(), stream_of(q))
    if codes is not out:
        out.copy_(codes)
    return out, out_scale


def paged_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                    kv_indices: torch.Tensor, kv_start: torch.Tensor, kv_len: torch.Tensor,
                    scale: float, out: Optional[torch.Tensor] = None,
                    group_prefix: Optional[torch.Tensor] = None, entries: Optional[int] = None) -> torch.Tensor:
    """softmax(q k^T * scale) v over each query token's slot list.

    q: [T, Hq, 128] bf16 (unit inner stride); k_cache / v_cache: [slots, Hk,
    128] float8_e4m3fn; kv_indices / kv_start / kv_len: int32 on the device.
    group_prefix: the plan of ``attention_plan`` for the same slot lists, or
    None (each call then finds the shared prefixes itself).  entries: the slots
    that the tokens' lists hold together, which decides over how many waves the
    keys of a query group are split (and so the order of its sums); without it
    the length of kv_indices is taken, and with a buffer longer than its lists
    the capacity counts.
    """
    T, Hq, D, slots, Hk = _check_attention_inputs(q, k_cache, v_cache, kv_indices, kv_start, kv_len)
    if out is None:
        out = torch.empty(T, Hq, D, dtype=torch.bfloat16, device=q.device)
    _attend(q, k_cache, v_cache, kv_indices, kv_start, kv_len, scale, out, _check_plan(group_prefix, T, Hq, Hk),
            _waves(T, Hq, Hk, kv_indices, entries))
    return out


def _attend(q, k_cache, v_cache, kv_indices, kv_start, kv_len, scale, out, plan: int, waves: int) -> None:
    """The launch, with inputs and plan checked."""
    T, Hq, D = q.shape
    slots, Hk, _ = k_cache.shape
    call("fr_paged_attention_split_fp8",
         q.data_ptr(), q.stride(0), q.stride(1),
         k_cache.data_ptr(), k_cache.stride(0), k_cache.stride(1),
         v_cache.data_ptr(), v_cache.stride(0), v_cache.stride(1),
         slots, kv_indices.data_ptr(), kv_start.data_ptr(), kv_len.data_ptr(),
         out.data_ptr(), out.stride(0), out.stride(1),
         T, Hq, Hk, D, float(scale), plan, waves, stream_of(q))
