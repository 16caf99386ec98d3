"""The transposing LDS reads of the GEMMs are written as instructions whose results arrive some instructions later
(csrc/gemm_common.h, tr_read / tr_wait): nothing but the compiler's own choice keeps it from copying, spilling or reusing such a
register before the wait.  So the assembly it makes of the file is read: from each read to the next wait for all LDS reads no
other instruction may name its registers, and no branch may come between."""
import os
import re
import subprocess

import pytest

from mycaffe_amd import build

READ, WAIT = "ds_read_b64_tr_b16", re.compile(r"s_waitcnt\b.*lgkmcnt\(0\)")


def registers(text):
    out = set()
    for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        out.update(range(int(a), int(b) + 1))
    return out | {int(a) for a in re.findall(r"\bv(\d+)\b", text)}


def check(lines):
    """(number of reads, list of violations) of one function's assembly."""
    pending, reads, bad = set(), 0, []
    for number, line in enumerate(lines):
        code = line.split(";")[0].strip()
        if not code or code.startswith((".", "#")) and not code.endswith(":"):
            continue
        if code.endswith(":") or code.startswith(("s_branch", "s_cbranch", "s_setpc", "s_swappc", "s_endpgm")):
            if pending:
                bad.append((number, code, sorted(pending)))
                pending = set()
            continue
        op, _, operands = code.partition(" ")
        if op == "s_waitcnt":
            if WAIT.match(code):
                pending = set()
            continue
        if op == READ:
            dst, _, rest = operands.strip().partition(",")
            hit = (registers(dst) | registers(rest)) & pending
            pending |= registers(dst)
            reads += 1
        else:
            hit = registers(operands) & pending
        if hit:
            bad.append((number, code, sorted(hit)))
    return reads, bad


def functions(assembly):
    name, body = None, []
    for line in assembly.splitlines():
        m = re.match(r"^(_Z\w+):", line)
        if m:
            name, body = m.group(1), []
        elif re.match(r"^\.Lfunc_end", line):
            if name:
                yield name, body
            name = None
        elif name:
            body.append(line)


def test_the_check_sees_what_it_should():
    good = ["ds_read_b64_tr_b16 v[2:3], v9 offset:64", "v_mfma_f32_32x32x16_bf16 v[20:35], v[4:7], v[8:11], v[20:35]", "s_waitcnt lgkmcnt(0)",
            "v_mov_b32_e32 v1, v2", ".LBB0_1:"]
    assert check(good) == (1, [])
    for wrong in ("v_mov_b32_e32 v1, v2", "v_add_u32_e32 v3, v4, v5", "ds_read_b64_tr_b16 v[3:4], v9", "s_cbranch_scc1 .LBB0_1", ".LBB0_2:",
                  "scratch_store_dwordx2 off, v[2:3], s0"):
        assert check([good[0], wrong] + good[2:])[1], wrong
    assert check([good[0], "s_waitcnt lgkmcnt(1)", "v_mov_b32_e32 v1, v2"])[1]


def test_no_instruction_touches_a_pending_read(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no compiler")
    out = str(tmp_path / "gemm_bf16.s")
    subprocess.run([build.HIPCC] + build.FLAGS + ["-w", "--cuda-device-only", "-S", os.path.join(build.CSRC, "gemm_bf16.hip"), "-o", out], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    with open(out) as f:
        found = [(name,) + check(body) for name, body in functions(f.read())]
    with_reads = [f for f in found if f[1]]
    assert len(with_reads) >= 21          # three layouts of seven tiles
    for name, reads, bad in with_reads:
        assert not bad, (name, bad[:5])


def test_no_instruction_touches_a_pending_read_of_the_split_fp32_kernel(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no compiler")
    out = str(tmp_path / "gemm_f32.s")
    subprocess.run([build.HIPCC] + build.FLAGS + ["-w", "--cuda-device-only", "-S", os.path.join(build.CSRC, "gemm_f32.hip"), "-o", out], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    with open(out) as f:
        found = [(name,) + check(body) for name, body in functions(f.read())]
    with_reads = [f for f in found if f[1]]
    assert len(with_reads) >= 18          # three layouts of six tiles
    for name, reads, bad in with_reads:
        assert not bad, (name, bad[:5])
