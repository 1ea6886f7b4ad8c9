"""Compile-time properties of the pipelined backward kernels, checked on their assembly.

Products that the dK / dV kernels at head dim 128 write as instructions:

The compiler does not see into these instructions, so it adds no wait states behind them: their result may be read by anything but the
next product on the same accumulator, or overwritten, twelve wait states later at the earliest (eight passes of a 32x32x16 product on
gfx950), and an operand written by the vector pipe may be read two wait states later (by another product: twelve).  This follows every
path from and to every such instruction and counts each instruction as one wait state (device side only, no GPU needed), in each of
the four builds that have them: registers are allocated, and instructions ordered, anew in each.

The stream of dQ: copies of the next tiles are on their way all the time and are waited for with a count, so nothing in it may wait for
a load of its own -- neither for a spilled register nor for one that the compiler believes still to be loading from the prologue.
"""
import concurrent.futures as cf
import os
import re
import subprocess

import pytest

from nvfuserexamples_amd import build as B

RESULT, OPERAND = 12, 2  # wait states
BUILDS = ["fmha_bwd_pipe_f16_d128", "fmha_bwd_pipe_bf16_d128", "fmha_bwd_pipe_f16_d128_strided", "fmha_bwd_pipe_bf16_d128_strided"]
STREAMS = BUILDS + ["fmha_bwd_pipe_f16_d64", "fmha_bwd_pipe_bf16_d64_strided"]


def registers(operand):
    m = re.fullmatch(r"([va])(?:\[(\d+):(\d+)\]|(\d+))", operand)
    if not m:
        return frozenset()
    lo, hi = (m[2], m[3]) if m[2] else (m[4], m[4])
    return frozenset((m[1], i) for i in range(int(lo), int(hi) + 1))


def parse(line):
    """(name, vector registers of each operand that has some, the operands) of an instruction, or None."""
    line = line.split(";")[0].strip()
    if not line or line.endswith(":") or line.startswith("."):
        return None
    name, _, rest = line.partition(" ")
    return name, [registers(o) for o in re.findall(r"[va]\[\d+:\d+\]|\b[va]\d+\b", rest)], [o.strip() for o in rest.split(",")]


def waits(ins):
    return int(ins[2][0], 0) + 1 if ins[0] == "s_nop" else 1


def written(ins):
    """Vector registers that an instruction of the vector or matrix pipe writes."""
    name, _, operands = ins
    if not name.startswith("v_"):
        return frozenset()
    return frozenset().union(*(registers(o) for o in operands[:2 if "swap" in name else 1]))


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
        name, regs, operands = ins
        if name == "s_endpgm":
            continue
        if name.startswith("v_mfma") and regs[0] == dst and not dst & (regs[1] | regs[2]):
            continue  # the next product of the chain
        if any(r & dst for r in regs):
            return i
        if name.startswith(("s_cbranch", "s_branch")):
            todo.append((labels[operands[0]], n + 1))
        if name != "s_branch":
            todo.append((i + 1, n + waits(ins)))
    return None


def predecessors(code, labels):
    """Line numbers that may be executed ahead of each line."""
    before = [[] for _ in code]
    for i, ins in enumerate(code):
        if ins and ins[0].startswith(("s_cbranch", "s_branch")):
            before[labels[ins[2][0]]].append(i)
        if i + 1 < len(code) and not (ins and ins[0] in ("s_branch", "s_endpgm")):
            before[i + 1].append(i)
    return before


def too_late(code, before, at):
    """The instruction that writes an operand of the product at `at` too shortly ahead of it, if there is one."""
    operands, seen, todo = code[at][1][1] | code[at][1][2], set(), [(i, 0) for i in before[at]]
    while todo:
        i, n = todo.pop()
        if n >= RESULT or (i, n) in seen:
            continue
        seen.add((i, n))
        ins = code[i]
        if ins is not None:
            if written(ins) & operands and n < (RESULT if ins[0].startswith("v_mfma") else OPERAND):
                return i
            n += waits(ins)
        todo += [(j, n) for j in before[i]]
    return None


def check(text):
    """Number of products written as instructions in a listing, and the first that breaks a rule: (its line, the other's)."""
    lines = text.split("\n")
    code = [parse(line) for line in lines]
    labels = {m[1]: i for i, line in enumerate(lines) if (m := re.match(r"(\.LBB\S+):", line))}
    before, inside, found = predecessors(code, labels), False, 0
    for i, line in enumerate(lines):
        if "#ASMSTART" in line:
            inside = True
        elif "#ASMEND" in line:
            inside = False
        elif inside and code[i] and code[i][0].startswith("v_mfma"):
            found += 1
            for j in (too_early(code, labels, i), too_late(code, before, i)):
                if j is not None:
                    return found, (line, lines[j])
    return found, None


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    at = tmp_path_factory.mktemp("asm")

    def compiled(name):
        src, _, defs = next(t for t in B._tus() if t[1] == name + ".o")
        out = str(at / (name + ".s"))
        subprocess.run([B.HIPCC, *B._flags(defs), "-S", "--cuda-device-only", os.path.join(B.CSRC, src), "-o", out], check=True,
                       capture_output=True)
        return open(out).read()

    with cf.ThreadPoolExecutor(len(STREAMS)) as ex:
        return dict(zip(STREAMS, ex.map(compiled, STREAMS)))


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("name", BUILDS)
def test_written_products_are_left_alone_until_they_are_done(name, listings):
    found, broken = check(listings[name])
    assert broken is None, broken
    assert found > 1000


def streams(text, kernel):
    """(function, lines) of the stream of every function of that name: the blocks that hold matrix instructions, of the innermost loop
    that copies and passes two barriers (two tiles a turn)."""
    lines, found = text.split("\n"), []
    for start in (i for i, line in enumerate(lines) if re.match(r"_Z\S*%s\S*:" % kernel, line)):
        body = lines[start:next(i for i in range(start, len(lines)) if lines[i].startswith(".Lfunc_end"))]
        labels = {m[1]: i for i, line in enumerate(body) if (m := re.match(r"(\.LBB\S+):", line))}
        spans = [(labels[m[1]], i) for i, line in enumerate(body) if (m := re.match(r"\s+s_c?branch\w*\s+(\.LBB\S+)", line)) and labels[m[1]] <= i]
        turns = []
        for a, b in spans:
            blocks, inside = [[]], False
            for line in body[a:b + 1]:
                if line.startswith(".LBB"):
                    blocks.append([])
                inside = "#ASMSTART" in line or (inside and "#ASMEND" not in line)
                blocks[-1].append((inside, line.split(";")[0].strip()))
                if re.match(r"\s+s_c?branch", line):
                    blocks.append([])
            blocks = [x for block in blocks if any(line.startswith("v_mfma") for _, line in block) for x in block]
            if sum("global_load_lds" in line for _, line in blocks) and sum("s_barrier" in line for _, line in blocks) >= 2:
                turns.append((a, b, blocks))
        found += [(body[0], blocks) for a, b, blocks in turns if not any((c, d) != (a, b) and a <= c and d <= b for c, d, _ in turns)]
    return found


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("name", STREAMS)
def test_streams_of_dq_wait_for_nothing_but_their_copies(name, listings):
    found = streams(listings[name], "fmha_bwd_dq_pipe_kernel")
    assert len({function for function, _ in found}) == 8  # no / per-key mask, causal or not, with dropout or not
    for function, lines in found:
        own = [line for inside, line in lines if not inside and ("vmcnt" in line or line.startswith("scratch_"))]
        assert not own, (function, own)


PRODUCT = "\t;#ASMSTART\n\tv_mfma_f32_32x32x16_f16 v[0:15], v[16:19], v[20:23], 0\n\t;#ASMEND\n"


@pytest.mark.parametrize("around,fine", [
    ("{}\ts_nop 11\n\tv_add_f32_e32 v30, v0, v31\n", True),
    ("{}\ts_nop 10\n\tv_add_f32_e32 v30, v0, v31\n", False),
    ("\tv_mov_b32_e32 v17, v40\n\ts_nop 1\n{}\ts_nop 15\n", True),
    ("\tv_mov_b32_e32 v17, v40\n\ts_nop 0\n{}\ts_nop 15\n", False),
    ("\tv_permlane32_swap_b32_e32 v40, v17\n{}\ts_nop 15\n", False),                           # the second register of a swap
    (".LBB0_1:\n{}\ts_nop 15\n\tv_mov_b32_e32 v21, v40\n\ts_cbranch_scc1 .LBB0_1\n", False),  # behind the loop's back edge
    (".LBB0_1:\n\ts_nop 1\n{}\ts_nop 15\n\tv_mov_b32_e32 v21, v40\n\ts_cbranch_scc1 .LBB0_1\n", True),
    ("\tv_mfma_f32_32x32x16_f16 v[16:31], v[40:43], v[44:47], 0\n\ts_nop 5\n{}\ts_nop 15\n", False),
    ("\tv_cmp_gt_f32_e32 vcc, v17, v18\n\tv_readfirstlane_b32 s3, v17\n{}\ts_nop 15\n", True),
])
def test_the_check_itself(around, fine):
    found, broken = check(around.format(PRODUCT) + "\ts_endpgm\n")
    assert found == 1 and (broken is None) == fine, broken
