"""What the kernel sources must say for the compiler to keep them right."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_inline_assembly_declares_the_registers_it_writes():
    # m0 is named in the text of an asm block and never an operand, so the
    # compiler learns only from the clobber list that it does not survive
    found = 0
    for path in glob.glob(os.path.join(ROOT, "ai-research_amd", "csrc", "**", "*.h*"), recursive=True):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for block in re.findall(r"\basm\b(?:\s+volatile)?\s*\((.*?)\)\s*;", text, flags=re.S):
            if re.search(r"\bs_mov_b32 m0\b", block):
                found += 1
                clobbers = block.rsplit(":", 1)[1]
                assert '"m0"' in clobbers, (os.path.basename(path), block)
    assert found > 0
