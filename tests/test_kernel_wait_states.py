"""Loads that go straight into LDS are written as asm, so the compiler does not keep the wait states that the hardware wants before
them.  Read from the disassembly of the built library: five between a vector instruction that writes a scalar register (a
readfirstlane, a reload of a spilled scalar) and a load that takes its offset or descriptor from it, one between a write of m0 and
a load that takes its target from there."""
import concurrent.futures
import os
import re
import shutil
import struct
import subprocess

import pytest

from deep8_amd import capi
from test_kernel_registers import _code_objects

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))
LOAD = re.compile(r"^\tbuffer_load[^/\n]* lds\b", re.M)
# instructions that may write a scalar register or m0: (opcode, first operands)
WRITER = re.compile(r"^\t(v_\S+ [^/\n]*?\bs[\d\[]|v_read[^/\n]*m0|s_\S+ m0\b)[^\n]*$", re.M)
INSTRUCTION = re.compile(r"^\t(\S+) ?([^/\n]*)// ([0-9A-F]+):", re.M)


def _scalars(operand):
    operand = operand.split()[0] if operand else ""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    return {operand} if operand == "m0" else {int(operand[1:])} if re.fullmatch(r"s\d+", operand) else set()


def _written(op, operands):
    if op.startswith(("v_add_co", "v_addc_co", "v_sub_co", "v_subb_co", "v_subrev", "v_subbrev", "v_mad_u64", "v_mad_i64", "v_div_scale")):
        return _scalars(operands[0]) | _scalars(operands[1])  # a carry
    return _scalars(operands[0])


def _too_soon(text, start, end, position, registers, states):
    """the loads into LDS that read `registers` within `states` wait states on any way on from `position`"""
    ways, found = [(position, 0)], []
    while ways:
        position, waited = ways.pop()
        while waited < states:
            m = INSTRUCTION.search(text, position, end)
            if not m:
                break
            op, operands, address = m[1], [o.strip() for o in m[2].split(",")], int(m[3], 16)
            position = m.end()
            if op.startswith("buffer_load") and operands[-1].endswith("lds") and registers & ({"m0"} | set().union(*map(_scalars, operands))):
                found.append(m[0].strip())
                break
            waited += int(operands[0], 0) + 1 if op == "s_nop" else 1
            if op == "s_branch" or op.startswith("s_cbranch"):
                offset = int(operands[0])
                target = text.find(f"// {address + 4 + 4 * (offset - 65536 if offset >= 32768 else offset):012X}:", start, end)
                assert target >= 0, m[0]
                ways.append((text.rfind("\n", 0, target) + 1, waited))
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                break
    return found


def _check(path):
    text = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
    loads = [m.start() for m in LOAD.finditer(text)]
    wrong, symbols = [], [m.start() for m in re.finditer(r"^[0-9a-f]+ <.*>:$", text, re.M)] + [len(text)]
    for start, end in zip(symbols, symbols[1:]):
        if not any(start < at < end for at in loads):
            continue
        for m in WRITER.finditer(text, start, end):
            i = INSTRUCTION.match(text, m.start())
            op, operands = i[1], [o.strip() for o in i[2].split(",")]
            registers = _written(op, operands)
            if registers:
                late = _too_soon(text, start, end, i.end(), registers, 1 if op.startswith("s_") else 5)
                wrong += [(text[start:text.index("\n", start)], i[0].strip(), l) for l in late]
    return len(loads), wrong


@pytest.mark.skipif(OBJDUMP is None, reason="llvm-objdump is not installed")
def test_loads_into_lds_wait_for_their_scalars(tmp_path):
    with open(capi.LIB_PATH, "rb") as f:
        blob = f.read()
    paths = []
    for at in _code_objects(blob):
        shoff, = struct.unpack_from("<Q", blob, at + 40)
        shentsize, shnum = struct.unpack_from("<HH", blob, at + 58)
        image = blob[at:at + shoff + shentsize * shnum]
        if b"gemm_tiled" in image or b"gemm_wide" in image:
            paths.append(tmp_path / f"{at}.elf")
            paths[-1].write_bytes(image)
    if not paths:
        pytest.skip("the library's code objects are compressed")
    with concurrent.futures.ProcessPoolExecutor(4) as pool:
        checked = list(pool.map(_check, paths))
    loads, wrong = sum(n for n, _ in checked), [w for _, some in checked for w in some]
    assert loads > 1000
    assert not wrong, f"{len(wrong)} of {loads} loads: {wrong[:3]}"
