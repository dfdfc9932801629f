"""Requests into LDS are written as assembly, which the compiler's hazard tables do not cover: a vector instruction that writes one of a
request's scalar operands needs five wait states in front of it, or the request goes out with what the register held before.  Nothing
in the source can promise that the compiler puts none there, so the objects that were built are read."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "relax_amd", "csrc")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
WAIT_STATES = 5


def scalars(operand):
    """The scalar registers that an operand names: 's[4:7]', 's8', 'm0', 'vcc', '-|s3|', ..."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return {"s%d" % i for i in range(int(m[1]), int(m[2]) + 1)}
    if operand in ("vcc", "exec"):
        return {operand + "_lo", operand + "_hi"}
    return {operand} if re.fullmatch(r"s\d+|m0|vcc_lo|vcc_hi|exec_lo|exec_hi", operand) else set()


def written_by_vector(op, operands):
    """What a vector instruction writes of the scalar registers: its first operand, and a carry behind the sum."""
    if not op.startswith("v_"):
        return set()
    written = scalars(operands[0]) if operands else set()
    if len(operands) > 1 and ("_co_" in op or op.startswith("v_div_scale")):
        written |= scalars(operands[1])
    if op.startswith("v_cmpx"):
        written |= scalars("exec")
    return written


def late_writes(lines):
    """(requests, [(the write, the request)]) of a listing: every path of fewer than five wait states that leads from a vector
    instruction's write to a request which reads it, along the branches as well."""
    code, at, sources = [], {}, {}
    for line in lines:
        m = re.match(r"\s+(\S+)(?:\s+(.*?))?\s*// ([0-9A-F]+):.*?(?:<\S+\+0x([0-9a-f]+)>)?\s*$", line)
        label = re.match(r"([0-9a-f]+) <", line)
        if label:
            base = int(label[1], 16)
        if not m:
            continue
        at[int(m[3], 16)] = len(code)
        operands = [o.strip() for o in re.split(r",\s*", re.sub(r"(\S)\s+(offen|off|offset|lds|glc|slc|nt|sc[01]|op_sel|dst_sel|quad_perm|row_).*", r"\1", m[2] or ""))]
        if m[1].startswith(("s_cbranch", "s_branch")) and m[4]:
            sources.setdefault(base + int(m[4], 16), []).append(len(code))
        code.append((m[1], operands, m[2] or "", int(m[3], 16)))
    came_from = {at[a]: froms for a, froms in sources.items() if a in at}
    requests, late = 0, []
    for i, (op, operands, text, _) in enumerate(code):
        if not (op.startswith("buffer_load") and re.search(r"\blds\b", text)):
            continue
        requests += 1
        reads = set().union(*(scalars(o) for o in operands)) | {"m0"}
        seen, todo = {}, [(i, 0, frozenset(reads))]
        while todo:
            j, states, live = todo.pop()
            before = ([j - 1] if j and code[j - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64") else []) + came_from.get(j, [])
            for b in before:
                bop, boperands, btext, _ = code[b]
                hit = written_by_vector(bop, boperands) & live
                if hit:
                    late.append((bop + " " + btext, op + " " + text))
                # (a scalar instruction that writes the register anew stands between)
                left = live - (set().union(*(scalars(o) for o in boperands[:1])) if bop.startswith("s_") and not bop.startswith("s_cmp") else set())
                passed = states + (int(boperands[0], 0) + 1 if bop == "s_nop" else 1)
                if passed < WAIT_STATES and left and seen.get((b, left), WAIT_STATES) > passed:
                    seen[(b, left)] = passed
                    todo.append((b, passed, left))
    return requests, late


def listing(path, tmp_path):
    shutil.copy(path, tmp_path / "o.o")
    subprocess.run([OBJDUMP, "--offloading", "o.o"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    device = [f for f in os.listdir(tmp_path) if f.startswith("o.o.") and "gfx950" in f]
    assert len(device) == 1, device
    return subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", device[0]], cwd=tmp_path, check=True, stdout=subprocess.PIPE, text=True).stdout.splitlines()


@pytest.mark.parametrize("name", ["wq_gemm_stream4.o", "wq_gemm_stream8.o", "wq_gemm_strip4.o", "wq_gemm_strip8.o"])
def test_no_vector_write_of_a_requests_scalar_operand_right_in_front_of_it(name, tmp_path):
    if not os.path.exists(os.path.join(CSRC, name)):
        subprocess.run(["make", "-C", CSRC, name], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    requests, late = late_writes(listing(os.path.join(CSRC, name), tmp_path))
    assert requests > 500
    assert not late, late[:5]


HEAD = "0000000000000100 <kernel>:"
REQUEST = ["\tbuffer_load_dwordx4 v1, s[4:7], s9 offen lds // 000000000300: 0"]


def numbered(lines, start):
    return ["\t%s // %012X: 0" % (line, start + 4 * i) for i, line in enumerate(lines)]


@pytest.mark.parametrize("lines,found", [
    (["v_readfirstlane_b32 s9, v2", "s_nop 0"], 1), (["v_readfirstlane_b32 s9, v2", "s_nop 3"], 1), (["v_readfirstlane_b32 s9, v2", "s_nop 4"], 0),
    (["v_readlane_b32 s6, v2, 3"] + ["v_mov_b32_e32 v3, v4"] * 4, 1), (["v_readlane_b32 s6, v2, 3"] + ["v_mov_b32_e32 v3, v4"] * 5, 0),
    (["v_readfirstlane_b32 m0, v2", "s_nop 0"], 1), (["v_readfirstlane_b32 s8, v2"], 0), (["v_cmp_eq_u32_e64 s[6:7], v1, v2"], 1),
    (["v_add_co_u32_e64 v1, s[8:9], v2, v3"], 1), (["v_readfirstlane_b32 s9, v2", "s_mov_b32 s9, s3"], 0), (["s_mov_b32 s9, s3"], 0)])
def test_the_reader_finds_what_it_looks_for(lines, found):
    requests, late = late_writes([HEAD] + numbered(lines, 0x300 - 4 * len(lines)) + REQUEST)
    assert requests == 1 and len(late) == found


def test_the_reader_follows_branches():
    branch = ["\tv_readfirstlane_b32 s9, v2 // 000000000100: 0", "\ts_branch 126 // 000000000104: 0 <kernel+0x200>", "\tv_mov_b32_e32 v3, v4 // 000000000108: 0"]
    assert len(late_writes([HEAD] + branch + REQUEST)[1]) == 1
    far = ["\tv_readfirstlane_b32 s9, v2 // 000000000100: 0", "\ts_endpgm // 000000000104: 0"]
    assert len(late_writes([HEAD] + far + REQUEST)[1]) == 0
