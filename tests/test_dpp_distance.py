"""Wait states before DPP reads, in the gfx950 assembly of the kernels that write
such instructions as inline statements (factor.hip, batched.hip).

The hardware wants two wait states between a vector instruction's write of a
register and a DPP read of it by another lane's instruction.  The compiler inserts
them only for instructions it has chosen itself; inline statements stand far enough
from the writes by the order of the source, which a change of it or of the register
allocation could undo without a wrong result on every run.  Every instruction counts
as one wait state, s_nop n as n + 1; both ways into a label are followed.
"""
import os
import re
import subprocess

import pytest

REG = re.compile(r"^v(?:(\d+)|\[(\d+):(\d+)\])$")


def _regs(operand):
    m = REG.match(operand.strip().split(" ")[0])
    if not m:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def close_reads(asm, need=2):
    """(line, text) of each DPP read too close behind a write of its register."""
    lines = []  # (number, label or None, mnemonic, operands)
    for no, text in enumerate(asm.splitlines(), 1):
        text = text.split(";")[0].split("//")[0].rstrip()
        label = re.match(r"^([.\w$]+):", text)
        if label:
            lines.append((no, label[1], None, []))
        elif re.match(r"^\s+[a-z]\w+", text):
            w = text.split(None, 1)
            lines.append((no, None, w[0], [o for o in w[1].split(",")] if len(w) > 1 else []))
    sources = {}
    for i, (_, label, op, args) in enumerate(lines):
        if op and op.startswith("s_cbranch") or op == "s_branch":
            sources.setdefault(args[-1].strip(), []).append(i)

    def written(i, regs, left, seen):
        # whether a vector instruction at most `left` wait states before line i writes one of regs
        while left > 0 and i > 0:
            i -= 1
            _, label, op, args = lines[i]
            if label:
                for b in sources.get(label, []):
                    if (b, left) not in seen and written(b + 1, regs, left, seen | {(b, left)}):
                        return True
                continue
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                return False
            if op.startswith("v_") and args and _regs(args[0]) & regs:
                return True
            left -= 1 + (int(args[0], 0) if op == "s_nop" else 0)
        return False

    bad, reads = [], 0
    for i, (no, label, op, args) in enumerate(lines):
        if op and op.endswith("_dpp") and len(args) > 1:
            reads += 1
            if written(i, _regs(args[1]), need, frozenset()):
                bad.append((no, op + " " + ",".join(args)))
    return bad, reads


def test_close_reads_are_found():
    far = "f:\n\tv_mul_f64 v[2:3], v[4:5], v[6:7]\n\ts_nop 1\n\tv_fmac_f64_dpp v[8:9], v[2:3], v[4:5] row_newbcast:0\n"
    near = far.replace("s_nop 1", "s_nop 0")
    loop = ("f:\n\tv_mov_b32 v9, 0\n.L1:\n\tv_fmac_f32_dpp v8, v3, v4 row_newbcast:1\n\tv_mov_b32 v5, 0\n"
            "\tv_mul_f32 v3, v3, v3\n\ts_cbranch_scc1 .L1\n")
    assert close_reads(far) == ([], 1)
    assert len(close_reads(near)[0]) == 1
    assert len(close_reads(loop)[0]) == 1
    assert close_reads(loop.replace("v_mul_f32 v3, v3", "v_mul_f32 v6, v3"))[0] == []


@pytest.mark.parametrize("source", ["factor.hip", "batched.hip"])
def test_reads_stand_two_wait_states_behind(source, tmp_path):
    from xkblas_amd import build as b
    out = str(tmp_path / "kernels.s")
    r = subprocess.run([b.HIPCC] + b.FLAGS + ["-x", "hip", "--cuda-device-only", "-S", os.path.join(b.CSRC, source), "-o", out],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    with open(out) as f:
        bad, reads = close_reads(f.read())
    assert reads > 100
    assert bad == []
