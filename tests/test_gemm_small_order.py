"""The counted waits of the K-split GEMM (gemm_fp8_small.hip) name the loads by
their number, in issue order: a slot's activation loads are waited for by letting
the later slots' loads stay in flight.  That holds only if no load of one ring
slot is issued among another slot's, which the compiler is free to do between
the slots of the prologue unless it is fenced.  Read off the compiled code."""

import re
import subprocess

import pytest

from flashrec_amd import build


@pytest.mark.skipif(not build.CSRC.is_dir(), reason="sources not present")
def test_prologue_issues_slot_by_slot(tmp_path):
    try:
        hipcc = build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    asm = tmp_path / "small.s"
    subprocess.run([hipcc, *build.HIPCC_FLAGS, "--offload-device-only", "-S", str(build.CSRC / "gemm_fp8_small.hip"),
                    "-o", str(asm)], check=True)
    seen = 0
    for args, body in re.findall(r"^_ZN2fr14gemm_fp8_smallI(\S+?)EEvNS_8GemmArgs\S*:\s[^\n]*\n(.*?)^\.Lfunc_end",
                                 asm.read_text(), re.S | re.M):
        fn, fm, _nw, ns = (int(x) for x in re.findall(r"Li(\d+)E", args))
        order = ""  # A: activation load to LDS, W: weight load, up to the first fragment read
        for line in body.splitlines():
            op = line.strip()
            if op.startswith("ds_read"):
                break
            if op.startswith("buffer_load"):
                order += "A" if op.endswith(" lds") else "W"
        # per slot 4 fm activation loads, then its 4 fn weight loads (each
        # perhaps twice, as two sides of a branch)
        want = ("A" * (4 * fm) + "W{%d,}" % (4 * fn)) * ns
        assert re.fullmatch(want, order), (args, order)
        seen += 1
    assert seen == 20
