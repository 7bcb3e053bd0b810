"""The 256 x 256 GEMM's LDS-DMAs, checked without a GPU."""

import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "primus-turbo_amd", "csrc")


def _asm_blocks(src):
    """The instructions of every inline-asm statement of a source text."""
    for m in re.finditer(r"asm volatile\(((?:\s*\"(?:[^\"\\]|\\.)*\")+)", src):
        text = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", m.group(1)))
        yield [i.strip() for i in text.replace("\\t", " ").split("\\n") if i.strip()]


def test_m0_is_written_an_instruction_ahead_of_the_dma_that_reads_it():
    """gfx950 needs one wait state between a scalar write of M0 and an LDS-DMA; the
    compiler, which adds it to its own code, does not look inside asm."""
    dmas = 0
    for name in sorted(os.listdir(CSRC)):
        for block in _asm_blocks(open(os.path.join(CSRC, name)).read()):
            for i, ins in enumerate(block):
                if not (ins.startswith("buffer_load") and ins.endswith(" lds")):
                    continue
                dmas += 1
                # M0 is written in the same statement, with an instruction between
                assert any(p.startswith("s_mov_b32 m0") for p in block[:i]), (name, block)
                assert not block[i - 1].startswith("s_mov_b32 m0"), (name, block)
    assert dmas >= 4
