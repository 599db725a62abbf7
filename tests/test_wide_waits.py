"""Refills of LDS under the wide prefill form's counted waits (prefill.hip),
read from the AMD assembly of the source: a direct load into LDS has no
register result, so nothing in the hardware holds it back until the reads of
the buffer it overwrites have returned.  LDS reads return in order, so at each
such load the reads still pending are those that no lgkmcnt wait covers yet.
The 6-bit form reads its words as 8-byte pieces and everything else as 16-byte
ones; the 4-bit form's words are 16-byte reads, as its fragments are, so for
it the number pending may not exceed the fragments of one step.  No GPU."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "pagedmoe_amd" / "csrc"
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-w", "-S",
         "--cuda-device-only", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _hipcc():
    return shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    if not _hipcc():
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("asm") / "prefill.s"
    subprocess.run([_hipcc(), *FLAGS, str(CSRC / "prefill.hip"), "-o", str(out)], check=True)
    return out.read_text()


def pending_at_lds_loads(body: str) -> list:
    """The LDS reads pending at each direct load, in program order."""
    pending, at = [], []
    for line in body.split("\n"):
        op = line.split(";")[0].split()
        if not op:
            continue
        if op[0].startswith("ds_read"):
            pending.append(op[0])
        wait = re.search(r"lgkmcnt\((\d+)\)", line)
        if op[0] == "s_waitcnt" and wait:
            n = int(wait.group(1))
            pending = pending[-n:] if n else []
        if op[0].startswith("global_load_lds"):
            at.append(list(pending))
    return at


@pytest.mark.parametrize("kernel", ["gateup_wide_kernel", "down_wide_kernel"])
@pytest.mark.parametrize("bits", [4, 6])
def test_no_word_read_pending_at_a_refill(asm, kernel, bits):
    found = re.search(rf"^_ZN\S*{kernel}ILi{bits}E\S*:", asm, re.M)
    assert found
    body = asm[found.start():asm.index(".Lfunc_end", found.start())]
    at = pending_at_lds_loads(body)
    assert len(at) > 40
    for pending in at:
        if bits == 6:
            assert all(op == "ds_read_b128" for op in pending), pending
        assert len(pending) <= 4, pending


def test_a_planted_refill_is_found():
    body = """
    ds_read_b64 v[0:1], v9
    ds_read_b64 v[2:3], v9 offset:8
    s_waitcnt lgkmcnt(1)
    global_load_lds_dwordx4 v8, s[0:1]
    """
    assert pending_at_lds_loads(body) == [["ds_read_b64"]]
