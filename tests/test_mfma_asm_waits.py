"""A compile-time property of the products that the dK / dV kernels at head dim 128 write as instructions, checked on their assembly.

The compiler does not see into these instructions, so it adds no wait states behind them: their result may be read by anything but the
next product on the same accumulator, or overwritten, twelve wait states later at the earliest (eight passes of a 32x32x16 product on
gfx950), and an operand written by the vector pipe may be read two wait states later.  This follows every path from every such
instruction and counts each instruction as one wait state (device side only, no GPU needed).
"""
import os
import re
import subprocess

import pytest

from nvfuserexamples_amd import build as B

RESULT, OPERAND = 12, 2  # wait states


def registers(operand):
    m = re.fullmatch(r"([va])(?:\[(\d+):(\d+)\]|(\d+))", operand)
    if not m:
        return frozenset()
    lo, hi = (m[2], m[3]) if m[2] else (m[4], m[4])
    return frozenset((m[1], i) for i in range(int(lo), int(hi) + 1))


def parse(line):
    line = line.split(";")[0].strip()
    if not line or line.endswith(":") or line.startswith("."):
        return None
    name, _, rest = line.partition(" ")
    return name, [registers(o) for o in re.findall(r"[va]\[\d+:\d+\]|\b[va]\d+\b", rest)], rest.split(",")[0].strip()


def waits(ins):
    return int(ins[2], 0) + 1 if ins[0] == "s_nop" else 1


def too_early(code, labels, at):
    """The instruction that touches the result of the product at `at` within its wait states, if there is one."""
    dst, seen, todo = code[at][1][0], set(), [(at + 1, 0)]
    while todo:
        i, n = todo.pop()
        if n >= RESULT or i >= len(code) or (i, n) in seen:
            continue
        seen.add((i, n))
        ins = code[i]
        if ins is None:
            todo.append((i + 1, n))
            continue
        name, regs, first = ins
        if name == "s_endpgm":
            continue
        if name.startswith("v_mfma") and regs[0] == dst and not dst & (regs[1] | regs[2]):
            continue  # the next product of the chain
        if any(r & dst for r in regs):
            return i
        if name.startswith(("s_cbranch", "s_branch")):
            todo.append((labels[first], n + 1))
        if name != "s_branch":
            todo.append((i + 1, n + waits(ins)))
    return None


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_written_products_are_left_alone_until_they_are_done(tmp_path):
    src, _, defs = next(t for t in B._tus() if t[1] == "fmha_bwd_pipe_f16_d128.o")
    out = str(tmp_path / "bwd.s")
    subprocess.run([B.HIPCC, *B._flags(defs), "-S", "--cuda-device-only", os.path.join(B.CSRC, src), "-o", out], check=True, capture_output=True)
    lines = open(out).read().split("\n")
    code = [parse(line) for line in lines]
    labels = {m[1]: i for i, line in enumerate(lines) if (m := re.match(r"(\.LBB\S+):", line))}
    written, found = False, 0
    for i, line in enumerate(lines):
        if "#ASMSTART" in line:
            written = True
        elif "#ASMEND" in line:
            written = False
        elif written and code[i] and code[i][0].startswith("v_mfma"):
            found += 1
            j = too_early(code, labels, i)
            assert j is None, (line, lines[j])
            n, k = 0, i - 1
            while n < OPERAND:
                if code[k]:
                    name, regs, _ = code[k]
                    writes = name.startswith("v_") and not name.startswith("v_mfma") and regs and regs[0] & (code[i][1][1] | code[i][1][2])
                    assert not writes, (lines[k], line)
                    n += waits(code[k])
                k -= 1
    assert found > 1000
