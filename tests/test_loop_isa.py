"""What the hand-counted K loops (onednn_amd/csrc/line_loops.hpp) rest on and the compiler does not know, read from the
instructions of the built kernel library:

  * the steady loops touch no scratch memory: a spilled register's reload waits for every load in flight;
  * MFMAs in inline assembly (the four-wavefront tiles): no vector instruction writes an operand in the two wait states
    before one, and nothing but an MFMA reads or overwrites an accumulator in the 18 wait states behind the one that writes
    it (more than any of the 16 x 16 shapes asks for)."""
import os
import re
import subprocess

import pytest

from onednn_amd import cabi

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
KERNEL = re.compile(r"^([0-9a-f]+) <(\S*(?:chain|f8|i8|mxf4)_gemm_kernel\S*)>:")
REG = re.compile(r"(?<![a-z0-9_])([va])(?:\[(\d+):(\d+)\]|(\d+))")


def regs(operand):
    out = set()
    for kind, lo, hi, one in REG.findall(operand):
        out |= {(kind, i) for i in range(int(lo or one), int(hi or one) + 1)}
    return out


def kernels(library, folder):
    """name -> [(address, mnemonic, operands, branch target or None)]"""
    lib = os.path.join(folder, "lib.so")
    os.symlink(os.path.abspath(library), lib)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=folder, check=True, capture_output=True)
    found = {}
    for f in sorted(os.listdir(folder)):
        if "gfx950" not in f:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], cwd=folder, check=True, capture_output=True, text=True).stdout
        body = base = None
        for line in text.splitlines():
            if line.endswith(">:"):
                m = KERNEL.match(line)
                body = found.setdefault(m.group(2), []) if m else None
                base = int(m.group(1), 16) if m else None
            elif body is not None and "//" in line:
                code, note = line.split("//", 1)
                op, _, rest = code.strip().partition(" ")
                at = int(note.split(":")[0], 16)
                to = re.search(r"\+0x([0-9a-f]+)>", note) if op.startswith(("s_branch", "s_cbranch")) else None
                body.append((at, op, rest.strip(), base + int(to.group(1), 16) if to else None))
    return found


@pytest.fixture(scope="module")
def tiles(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    found = kernels(cabi.KERNEL_LIB_PATH, str(tmp_path_factory.mktemp("isa")))
    found = {k: v for k, v in found.items() if "f32_mma" not in k}  # (the plain loop)
    assert len(found) >= 40
    return found


def is_mfma(op):
    return op.startswith("v_mfma")


def steady_loop(code):
    """the first loop with MFMAs: the steps inside K, two to a round"""
    at = {a: i for i, (a, *_) in enumerate(code)}
    for i, (_, _, _, to) in enumerate(code):
        if to is not None and to in at and at[to] < i:
            body = code[at[to]:i + 1]
            if sum(is_mfma(op) for _, op, *_ in body) >= 32:
                return body
    return None


def test_steady_loops_are_free_of_scratch_memory(tiles):
    for name, code in tiles.items():
        loop = steady_loop(code)
        assert loop, name
        spills = [op for _, op, *_ in loop if op.startswith("scratch_")]
        assert not spills, (name, spills)


def hazards(code):
    bad = []
    window = []  # (wait states since, registers written) of the last vector instructions
    accs = {}    # accumulator register -> wait states since the MFMA that wrote it
    for at, op, rest, _ in code:
        if op in ("s_branch", "s_endpgm"):  # what stands behind is reached from elsewhere
            window, accs = [], {}
            continue
        states = 1 + int(rest, 0) if op == "s_nop" else 1
        operands = [x.strip() for x in re.split(r",(?![^\[]*\])", rest)] if rest else []
        if is_mfma(op):
            need = set().union(*(regs(x) for x in operands[1:6]))
            if any(age < 2 and written & need for age, written in window):
                bad.append((hex(at), op, rest))
        elif op.startswith("v_"):
            wait = {r: n for r, n in accs.items() if n < 18}
            if wait and set(wait) & set().union(*(regs(x) for x in operands)):
                bad.append((hex(at), op, rest))
        window = [(age + states, w) for age, w in window if age + states < 2]
        accs = {r: n + states for r, n in accs.items() if n + states < 18}
        if is_mfma(op):
            accs.update(dict.fromkeys(regs(operands[0]), 0))
        elif op.startswith("v_") and operands:
            window.append((0, regs(operands[0])))
    return bad


def test_wait_states_around_inline_matrix_instructions(tiles):
    narrow = {k: v for k, v in tiles.items() if "geo_tILi4ELi128E" in k}
    assert len(narrow) >= 15
    for name, code in narrow.items():
        assert not hazards(code), (name, hazards(code)[:3])


def test_the_check_finds_planted_hazards():
    mfma = (8, "v_mfma_f32_16x16x32_bf16", "a[0:3], v[4:7], v[8:11], a[0:3]", None)
    nop = (4, "s_nop", "1", None)
    write = (0, "v_xor_b32_e32", "v5, v1, v2", None)
    read = (12, "v_accvgpr_read_b32", "v1, a2", None)
    assert hazards([write, mfma]) and not hazards([write, nop, mfma])
    assert hazards([mfma, read]) and not hazards([mfma, (9, "s_nop", "15", None), nop, read])
