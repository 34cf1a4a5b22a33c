"""CPU test of the inline assembly that moves memory into LDS: the compiler does not look into an asm block, so the wait states that the
instruction set asks for have to stand in the text."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vox_serve_amd", "csrc")
ASM = re.compile(r"asm\s+volatile\s*\((.*?)\)\s*;", re.S)


def lds_dma_blocks():
    out = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        with open(path) as f:
            for m in ASM.finditer(f.read()):
                text = "".join(re.findall(r'"([^"]*)"', m.group(1).split(":")[0])).replace("\\n\\t", "\n").split("\n")
                if any("load_lds" in t for t in text):
                    out.append(pytest.param(text, m.group(1), id=f"{os.path.basename(path)}-{len(out)}"))
    return out


BLOCKS = lds_dma_blocks()
assert BLOCKS


def wait_states(lines):
    """An instruction is one, s_nop N is N + 1."""
    return sum(int(t.split()[1]) + 1 if t.startswith("s_nop") else 1 for t in lines)


@pytest.mark.parametrize("text,source", BLOCKS)
def test_m0_is_settled_when_the_dma_reads_it(text, source):
    """A scalar write of m0, then one wait state, then the instruction that takes its LDS address from m0; and the block says that it writes m0."""
    load = next(i for i, t in enumerate(text) if "load_lds" in t)
    wrote = next(i for i, t in enumerate(text) if re.match(r"s_\w+ m0,", t))
    assert wrote < load and wait_states(text[wrote + 1:load]) >= 1
    assert '"m0"' in source


@pytest.mark.parametrize("text,source", BLOCKS)
def test_a_scalar_base_is_settled_when_the_dma_reads_it(text, source):
    """The base comes from outside the block, where v_readfirstlane or v_readlane may have written it last: five wait states between a vector
    write of a scalar register and the memory instruction that addresses with it."""
    load = next(i for i, t in enumerate(text) if "load_lds" in t)
    if not text[load].endswith("off"):
        assert wait_states(text[:load]) >= 5
