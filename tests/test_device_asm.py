"""What the gfx950 assembly of this build's kernels must hold where the
compiler does not see to it: inside inline asm no wait state is added."""
import glob
import os
import re
import subprocess

import pytest

from gsdlq import build

SOURCES = [s for s in sorted(glob.glob(os.path.join(build.CSRC, "*.hip"))) if re.search(r"load_lds", open(s).read())]
LDS_LOAD = re.compile(r"(global|buffer|scratch)_load_lds_|buffer_load_.*\blds\b")
M0_WRITE = re.compile(r"s_\w+\s+m0\b")


def _unwaited(lines):
    """The loads to LDS whose last instruction in text order (labels and
    directives aside) wrote m0."""
    bad, last = [], ""
    for n, line in enumerate(lines, 1):
        ins = line.split(";")[0].strip()
        if not ins or ins.startswith(".") or ins.endswith(":"):
            continue
        if LDS_LOAD.match(ins) and M0_WRITE.match(last):
            bad.append((n, last, ins))
        last = ins
    return bad


def test_unwaited_finds_the_form():
    load = "global_load_lds_dwordx4 v[2:3], off"
    assert _unwaited(["\ts_mov_b32 m0, s16", "\t;;#ASMEND", ".LBB0_1:", "\t" + load])
    assert not _unwaited(["\ts_mov_b32 m0, s16", "\ts_nop 0", "\t" + load])


@pytest.mark.parametrize("src", SOURCES, ids=os.path.basename)
def test_lds_loads_wait_for_m0(src, tmp_path):
    """One wait state between a scalar write of m0 and a load to LDS."""
    out = tmp_path / "device.s"
    subprocess.run([build._hipcc()] + build.HIPCC_FLAGS + ["--cuda-device-only", "-S", src, "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    lines = out.read_text().splitlines()
    assert any(LDS_LOAD.match(line.strip()) for line in lines)
    assert not _unwaited(lines)
