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
    """M0 is written by the copies' asm alone (the compiler does not track it across one), never in the instruction
    before the copy."""
    copies = 0
    for name, ins in kernels.items():
        for before, now in zip(ins, ins[1:]):
            assert "m0" not in now[1] or (now[2] and now[0] == "s_mov_b32"), f"{name}: {now[3]}"
            if "_load_lds_" in now[0]:
                copies += 1
                assert before[1][:1] != ["m0"], f"{name}: {before[3]} directly before {now[3]}"
    assert copies


def _registers(operand):
    kind, span = operand[0], operand[1:].strip("[]").split(":")
    return {(kind, r) for r in range(int(span[0]), int(span[-1]) + 1)}


def test_no_asm_leaves_a_global_load_into_registers_in_flight(kernels):
    """The compiler takes an asm's outputs as written: a global load there either goes to LDS or is waited for there."""
    for name, ins in kernels.items():
        for i, (op, _, in_asm, text) in enumerate(ins):
            if in_asm and op.startswith(("global_load_dword", "buffer_load_dword")):
                rest = ins[i + 1:]
                end = next(j for j, step in enumerate(rest) if not step[2])
                assert any(step[0] == "s_waitcnt" and "vmcnt(0)" in step[3] for step in rest[:end]), f"{name}: {text}"


def test_registers_of_asm_lds_reads_are_untouched_until_their_wait(kernels):
    """In program order, no instruction names a register that an LDS read issued by an asm may still write."""
    for name, ins in kernels.items():
        flight = []  # LDS instructions not waited for: (registers an asm read writes, text)
        for op, operands, in_asm, text in ins:
            if op == "s_waitcnt":
                count = re.search(r"lgkmcnt\((\d+)\)", text)
                if count:
                    flight = flight[max(0, len(flight) - int(count[1])):] if int(count[1]) else []
                continue
            named = set().union(*map(_registers, operands)) if operands else set()
            hit = next((read for regs, read in flight if regs & named), None)
            assert hit is None, f"{name}: {text} while {hit} is in flight"
            if op.startswith("ds_"):
                flight.append((_registers(operands[0]) if in_asm and op.startswith("ds_read") else set(), text))
