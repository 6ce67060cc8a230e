"""What the kernels' inline assembly may hold, read from the sources (no GPU).

Inside an asm statement, and between it and what stands in front of it, the compiler puts no wait states: a vector instruction that reads a condition (vcc or a pair of scalar registers) which
a vector instruction wrote needs two of them on gfx950, a reader of a matrix result as many as that product still runs, and none of it shows in a result until a schedule changes.  So vector
arithmetic is left to the compiler; asm statements hold waits, requests to memory and what addresses them."""
import glob
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNELS = sorted(glob.glob(os.path.join(ROOT, "nano-vllm-rs_amd", "csrc", "kernels", "*.h*")))


def _statements(text):
    """The instructions of every asm statement: the string literals in front of its first operand list."""
    for m in re.finditer(r'\basm\s*(?:volatile\s*)?\(((?:\s*"(?:[^"\\]|\\.)*")+)', text):
        literals = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', m.group(1)))
        yield text.count("\n", 0, m.start()) + 1, [i.strip() for i in re.split(r"\\n|\\t|;", literals) if i.strip()]


def test_scan_sees_every_instruction():
    text = 'asm volatile("s_mov_b32 m0, %0\\n\\ts_nop 0\\n\\t"\n    "global_load_lds_dwordx4 %1, off" : : "s"(a), "v"(b)); asm("" : "+v"(x)); asm("v_cmp_gt_i32 vcc, %1, %2" : );'
    assert [i for _, i in _statements(text)] == [["s_mov_b32 m0, %0", "s_nop 0", "global_load_lds_dwordx4 %1, off"], [], ["v_cmp_gt_i32 vcc, %1, %2"]]


@pytest.mark.parametrize("path", KERNELS, ids=[os.path.basename(p) for p in KERNELS])
def test_inline_assembly_holds_no_vector_arithmetic(path):
    with open(path) as f:
        text = f.read()
    for line, instructions in _statements(text):
        for at, i in enumerate(instructions):
            assert not i.startswith("v_"), "%s:%d: %s" % (path, line, i)
            if i.split()[0] in ("s_mov_b32", "s_add_u32") and i.split()[1] == "m0,":       # a request into LDS reads m0 one wait state behind its write at the earliest
                following = instructions[at + 1:at + 2]
                assert not following or not following[0].startswith("global_load_lds"), "%s:%d: %s" % (path, line, i)


def _whole(text):
    """Every asm statement with its operands."""
    for m in re.finditer(r'\basm\s*(?:volatile\s*)?\(', text):
        depth, at, quoted = 1, m.end(), False
        while depth:
            c = text[at]
            if quoted and c == "\\":
                at += 1
            elif c == '"':
                quoted = not quoted
            elif not quoted:
                depth += {"(": 1, ")": -1}.get(c, 0)
            at += 1
        yield text.count("\n", 0, m.start()) + 1, text[m.start():at]


@pytest.mark.parametrize("path", KERNELS, ids=[os.path.basename(p) for p in KERNELS])
def test_inline_assembly_tells_the_compiler_of_m0(path):
    """A request into LDS takes its place from M0: the statement sets M0 itself and puts back what it held, or M0 goes in and out as an operand, so that the compiler keeps nothing else there."""
    with open(path) as f:
        text = f.read()
    for line, statement in _whole(text):
        instructions = next(i for _, i in _statements(statement))
        writes = [at for at, i in enumerate(instructions) if re.match(r"s_\w+ m0,", i)]
        if writes and not re.search(r'"(=\{m0\}|m0)"', statement):
            kept = [i.split()[1].rstrip(",") for i in instructions[:writes[0]] if re.match(r"s_mov_b32 %\d+, m0$", i)]
            assert kept and instructions[writes[-1]] == "s_mov_b32 m0, " + kept[0], "%s:%d: M0 written" % (path, line)
        for at, i in enumerate(instructions):
            if i.startswith("global_load_lds"):
                assert '"{m0}"' in statement or (writes and writes[0] < at), "%s:%d: M0 read" % (path, line)
