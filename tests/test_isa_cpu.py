"""Hazards that inline asm brings and the compiler does not resolve, checked on the gfx950 assembly that hipcc makes of
this repository's sources (no GPU)."""
import re
import subprocess

import pytest

from fastdecisions_amd import _build

SOURCES = [s for s in _build.SOURCES if s.endswith(".hip") and "load_lds" in (_build.CSRC / s).read_text()]


@pytest.fixture(scope="module", params=SOURCES)
def kernels(request):
    """{function: [(opcode, register operands, inside an asm block, text)]} in program order."""
    out = subprocess.run([_build.hipcc(), *_build.COMMON_FLAGS, "-x", "hip", *_build.DEVICE_FLAGS, "--cuda-device-only",
                          "-S", str(_build.CSRC / request.param), "-o", "-"], check=True, capture_output=True, text=True)
    found, current, in_asm = {}, None, False
    for line in out.stdout.splitlines():
        name = re.match(r"(_Z\w+):", line)
        if name:
            current = found.setdefault(name[1], [])
        elif "#ASMSTART" in line or "#ASMEND" in line:
            in_asm = "#ASMSTART" in line
        else:
            text = line.split(";")[0].strip()
            if current is not None and text and not text.startswith(".") and not text.endswith(":"):
                op, _, rest = text.partition(" ")
                current.append((op, re.findall(r"[vsa]\[\d+:\d+\]|\b[vsa]\d+\b|\bm0\b", rest), in_asm, text))
    found = {name: ins for name, ins in found.items() if ins}
    assert found
    return found


def test_a_wait_state_between_m0_and_the_copy_that_reads_it(kernels):
    copies = 0
    for name, ins in kernels.items():
        for before, now in zip(ins, ins[1:]):
            if "_load_lds_" in now[0]:
                copies += 1
                assert before[1][:1] != ["m0"], f"{name}: {before[3]} directly before {now[3]}"
    assert copies
