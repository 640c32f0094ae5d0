"""Properties of the compiled kernels that only their assembly shows (no GPU:
the sources are compiled for gfx950 here)."""

import os
import re
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

CSRC = os.path.join(ROOT, "mini-tp_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def _assembly(source: str, out: str) -> list[str]:
    flags = subprocess.run(["make", "-pn", "-C", CSRC], capture_output=True, text=True).stdout
    flags = re.search(r"^FLAGS := (.*)$", flags, re.M).group(1).replace("$(ARCH)", "gfx950").replace("$(EXTRA)", "")
    subprocess.run([HIPCC, *flags.split(), "-w", "-x", "hip", "--cuda-device-only", "-S", source, "-o", out], cwd=CSRC,
                   check=True)
    lines = (ln.split(";")[0].strip() for ln in open(out))
    # instructions only (no directives, no labels)
    return [ln for ln in lines if ln and not ln.startswith((".", "//")) and not ln.endswith(":")]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("source", ["gemm.hip", "gemm_tile.hip"])
def test_a_load_to_lds_never_follows_the_write_of_m0_directly(source, tmp_path):
    """m0 holds the LDS address of a buffer load to LDS; gfx9 hardware needs one wait state
    between a scalar write of m0 and such a load, and the compiler adds none
    in front of inline assembly."""
    code = _assembly(source, str(tmp_path / "out.asm"))
    loads = [i for i, ins in enumerate(code) if re.match(r"buffer_load_\w+ .*\blds$", ins)]
    assert loads
    bad = [code[i - 1:i + 1] for i in loads if re.match(r"[sv]_\w+ m0,", code[i - 1])]
    assert not bad, bad[:3]
    # the same for scalar registers that a vector instruction wrote: five wait
    # states before a vector memory instruction reads them
    for i in loads:
        read = set()
        for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", code[i]):
            read |= set(range(int(lo), int(hi) + 1))
        read |= {int(r) for r in re.findall(r"\bs(\d+)\b", code[i])}
        for ins in code[max(i - 5, 0):i]:
            wrote = re.match(r"v_read(?:first)?lane_b32 s(\d+),", ins)
            assert not (wrote and int(wrote.group(1)) in read), (ins, code[i])
