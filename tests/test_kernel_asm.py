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
