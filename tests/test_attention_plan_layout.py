"""CPU checks of the attention plan's layout: where a group's record stands
depends on the group alone, and a walk over its segments ends and takes every
token once for any call, whatever the plan was made for."""

import shutil
import subprocess
from pathlib import Path

import pytest
import torch

HERE = Path(__file__).resolve().parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_record_walks(tmp_path):
    exe = tmp_path / "attn_plan_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", str(HERE.parent / "flashrec_amd" / "csrc"),
                    "-o", str(exe), str(HERE / "csrc" / "attn_plan_check.cc")], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split("=")[1]) > 10000


@pytest.mark.parametrize("hq,hk", [(16, 8), (8, 8), (16, 4), (16, 2)])
def test_plan_size_is_whole_records(hq, hk):
    """All token counts of a group need the same room, and n groups n times it."""
    from flashrec_amd.attention import plan_size

    tok = 32 // (hq // hk)
    one = plan_size(1, hq, hk)
    assert one > 2 * tok
    for t in (1, tok - 1, tok, tok + 1, 3 * tok - 1, 40 * tok):
        assert plan_size(t, hq, hk) == -(-t // tok) * one
    assert plan_size(0, hq, hk) == 0


def test_what_a_plan_may_be():
    """Views of whole records and flat buffers of them, bare prefixes, and what is refused."""
    from flashrec_amd.attention import paged

    groups, stride = paged._groups(64, 16, 8)
    assert groups == 4 and stride == paged.plan_size(1, 16, 8)
    flat = torch.zeros(4 * stride, dtype=torch.int32)
    rows = paged._plan_rows(flat, 64, 16, 8)
    assert rows.shape == (4,) and rows.data_ptr() == flat.data_ptr()
    assert paged._plan_records(rows, 4, stride) and paged._plan_records(rows, 3, stride)
    assert paged._plan_records(flat, 4, stride) and paged._plan_records(rows[1:], 3, stride)
    assert not paged._plan_records(rows, 5, stride)
    assert not paged._plan_records(flat[: 4 * stride - 1], 4, stride)
    # a view whose last record would pass the end of its storage
    assert not paged._plan_records(flat[stride - 1:].as_strided((4,), (stride,), 0), 5, stride)
    assert not paged._plan_records(torch.zeros(3 * stride + 1, dtype=torch.int32)[::stride], 4, stride)
    for bad in (rows[:-1], torch.zeros(3, dtype=torch.int32), torch.zeros(4, dtype=torch.int64),
                torch.zeros(8, dtype=torch.int32)[::2]):
        with pytest.raises(ValueError, match="plan"):
            paged._check_plan_buffer(bad, 4, paged._plan_records(bad, 4, stride))


def test_split_of_prompts_over_cached_prefixes():
    """A prompt that continues a long cached prefix is split like one without;
    prompts of a token each are split as decode rows are."""
    from types import SimpleNamespace

    from flashrec_amd._lib import load
    from flashrec_amd.attention.paged import AttentionBackend

    be = AttentionBackend(SimpleNamespace(device=torch.device("cpu")), 16, 8, 128)

    def waves(prompts):  # (cached, new) of each
        seq = torch.tensor([c + e for c, e in prompts], dtype=torch.int32)
        plan = be._plan_prefill(SimpleNamespace(
            n_rows=len(prompts), seq_lens_cpu=seq, extend_seq_lens=[e for _, e in prompts],
            extend_prefix_lens=[c for c, _ in prompts], kv_indices=torch.zeros(int(seq.sum()), dtype=torch.int32)))
        return load().fr_paged_attention_waves(int(plan["start"].numel()), 16, 8, plan["entries"])

    assert waves([(0, 100)]) == waves([(1500, 100)])
    assert waves([(0, 1100)]) == waves([(9000, 1100)]) > 1
    assert waves([(0, 300)] * 4) == waves([(3000, 300)] * 4) > 1
    assert waves([(129, 1)] * 2048) == load().fr_paged_attention_waves(2048, 16, 8, 2048 * 130)


def test_rows_of_one_head_group_are_split():
    from flashrec_amd._lib import load

    w = load().fr_paged_attention_waves
    assert w(1024, 32, 32, 1024 * 200) == 2 and w(2048, 16, 8, 2048 * 130) == 1
