"""CPU: what the kernels' inline assembly may hold.  The compiler inserts the wait states between a matrix instruction and a reader of its
result, but not in front of an asm statement, which it does not look into; and it knows of the registers a statement writes from its
operands alone."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-candle_amd", "csrc")


def asm_statements():
    """(file, line, text between the parentheses) of every asm statement"""
    out = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        src = open(path).read()
        for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(", src):
            depth, i = 1, m.end()
            while depth:
                depth += {"(": 1, ")": -1}.get(src[i], 0)
                i += 1
            out.append((os.path.basename(path), src.count("\n", 0, m.start()) + 1, src[m.end():i - 1]))
    return out


def templates(text):
    """the instructions: string literals before the first operand list"""
    return "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', re.split(r'"\s*:', text, maxsplit=1)[0] + '"')).replace("\\n\\t", "\n")


def test_the_statements_are_found():
    found = asm_statements()
    assert len(found) > 20 and any("ds_read_b128" in templates(t) for _, _, t in found)


@pytest.mark.parametrize("where", asm_statements(), ids=lambda w: f"{w[0]}:{w[1]}")
def test_no_vector_arithmetic(where):
    # a vector instruction in asm may read a matrix result before its wait states are over
    assert not re.search(r"\bv_\w+", templates(where[2])), where


@pytest.mark.parametrize("where", asm_statements(), ids=lambda w: f"{w[0]}:{w[1]}")
def test_no_register_is_written_behind_the_compilers_back(where):
    # M0 above all: the LDS-DMA builtin and indexed registers read it, set up wherever the compiler likes
    assert not re.search(r"\bs_\w+\s+m0\b", templates(where[2])), where
