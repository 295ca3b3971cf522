"""The matrix instructions of the built kernels against the hardware's rule for their operands, read from the
disassembly of the library that was built here.

A VALU instruction that writes a register needs two wait states (instructions, or the count of an s_nop)
before an MFMA that reads it.  The compiler keeps that for its own MFMAs; the e2m1 ones of the tiled GEMM are
inline assembly, which its hazard pass does not look into, so the source has to keep the distance."""
import re
import subprocess
from pathlib import Path

import pytest

from driss_torch_amd import cabi

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
WAIT_STATES = 2  # VALU write of a VGPR or AGPR -> MFMA read

_REGS = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")


def _regs(operand):
    """registers of one operand, as (file, number) pairs"""
    m = _REGS.match(operand.strip().lstrip("-|"))
    if not m:
        return set()
    lo, hi = (int(m[2]), int(m[2])) if m[2] else (int(m[3]), int(m[4]))
    return {(m[1], n) for n in range(lo, hi + 1)}


def _operands(text):
    """the operand list of an instruction: split at commas outside brackets"""
    parts = text.split(None, 1)
    return re.split(r",\s*(?![^\[]*\])", parts[1]) if len(parts) > 1 else []


def _functions(listing):
    """{name: [(address, text, target address or None)]}"""
    out, name, base = {}, None, {}
    for line in listing.splitlines():
        head = re.match(r"([0-9a-f]+) <(.+)>:$", line)
        if head:
            name = head[2]
            base[name] = int(head[1], 16)
            out[name] = []
            continue
        body = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):[ 0-9A-F]*(?:<(.+?)(?:\+0x([0-9a-f]+))?>)?$", line)
        if name and body:
            target = base[body[3]] + int(body[4] or "0", 16) if body[3] in base else None
            out[name].append((int(body[2], 16), body[1], target))
    return out


def violations(code):
    """(position, MFMA, VALU instruction, distance) wherever a VALU write is fewer than WAIT_STATES in front of
    an MFMA that reads the register, along any path through the function"""
    at = {address: i for i, (address, _, _) in enumerate(code)}
    jumps = {}
    for i, (_, text, target) in enumerate(code):
        if target in at and text.startswith(("s_branch", "s_cbranch")):
            jumps.setdefault(at[target], []).append(i)

    def predecessors(i):
        if i and not code[i - 1][1].startswith(("s_branch", "s_endpgm", "s_setpc")):
            yield i - 1
        yield from jumps.get(i, [])

    found = []
    for i, (_, text, _) in enumerate(code):
        if not text.startswith("v_mfma"):
            continue
        read = set().union(*(_regs(o) for o in _operands(text)[1:]))
        open_paths = [(p, 0) for p in predecessors(i)]
        while open_paths:
            p, states = open_paths.pop()
            before = code[p][1]
            if before.startswith("v_") and not before.startswith("v_mfma"):
                ops = _operands(before)
                written = _regs(ops[0]) if ops else set()
                if before.startswith("v_swap"):
                    written |= _regs(ops[1])
                if written & read:
                    found.append((i, text, before, states))
            states += int(before.split()[1], 0) + 1 if before.startswith("s_nop") else 1
            if states < WAIT_STATES:
                open_paths += [(q, states) for q in predecessors(p)]
    return found


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: code} of every kernel with an MFMA in the built library"""
    where = tmp_path_factory.mktemp("code")
    lib = where / "lib.so"
    lib.write_bytes(Path(cabi._LIB_PATH).read_bytes())
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=where)
    found = {}
    for obj in sorted(where.glob("*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True, text=True).stdout
        if "v_mfma" in text:
            found.update({k: c for k, c in _functions(text).items() if any(t.startswith("v_mfma") for _, t, _ in c)})
    return found


def test_checker_sees_a_short_distance():
    mfma = "v_mfma_scale_f32_16x16x128_f8f6f4 a[0:3], v[20:23], v[84:87], a[0:3], v52, v196 op_sel_hi:[0,0,0] cbsz:4 blgp:4"

    def listing(*instructions):
        return _functions("0000000000001000 <k>:\n" + "".join(f"\t{t}  // {0x1000 + 4 * i:012X}: 00000000\n"
                                                              for i, t in enumerate(instructions)))["k"]

    for write in ("v_accvgpr_mov_b32 a3, a80", "v_and_b32_e32 v196, s4, v7", "v_mov_b32_e32 v85, v1"):
        assert len(violations(listing(write, mfma))) == 1
        assert len(violations(listing(write, "s_nop 0", mfma))) == 1
        assert not violations(listing(write, "s_nop 1", mfma))
        assert not violations(listing(write, "s_barrier", "s_waitcnt lgkmcnt(0)", mfma))
    assert not violations(listing("v_and_b32_e32 v195, s4, v196", mfma))  # writes nothing that is read
    # round a loop: the write at its end, the MFMA at its head
    loop = _functions("0000000000001000 <k>:\n\ts_nop 7 // 000000001000: 00\n\t" + mfma + " // 000000001004: 00\n"
                      "\tv_mov_b32_e32 v52, v1 // 00000000100C: 00\n\ts_cbranch_scc1 65533 // 000000001010: 00 <k+0x4>\n"
                      "\ts_endpgm // 000000001014: 00\n")["k"]
    assert [v[0] for v in violations(loop)] == [1]


def test_every_mfma_is_two_wait_states_behind_the_valu_writes_of_its_operands(kernels):
    assert sum(len(c) for c in kernels.values()) > 10000 and any("mx_gemm" in k for k in kernels)
    bad = {k: v for k, c in kernels.items() if (v := violations(c))}
    report = "\n".join(f"{k}: {len(v)}, e.g. '{v[0][2]}' {v[0][3]} before '{v[0][1]}'" for k, v in bad.items())
    assert not bad, report
