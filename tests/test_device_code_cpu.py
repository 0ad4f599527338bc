"""Properties of the device code that a run on the GPU cannot show, checked on
its source and on the listing of the built library (no GPU calls)."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "matrixalgebrakit.jl_amd" / "csrc"


def body(source, head):
    """The text of the function whose definition contains `head`, braces included."""
    at = source.index("{", source.index(head))
    depth = 0
    for i in range(at, len(source)):
        depth += {"{": 1, "}": -1}.get(source[i], 0)
        if depth == 0:
            return source[at:i + 1]
    raise AssertionError(head)


def test_factor_step_reads_a_blocks_state_once():
    """A task of the batched factorisation may store the state word of a block
    while the block's other tasks of the same launch start: all threads of a
    workgroup must take the same exit, or some waves leave before its barriers
    and the others go on without what those waves would have loaded.  So one
    thread reads the word, and every access to it is atomic."""
    text = body((CSRC / "mak_bchol.hip").read_text(), "bchol_factor_kernel(const BCholProb* P")
    uses = [line.strip() for line in text.splitlines() if "p.state" in line]
    assert len(uses) == 2 and all("__hip_atomic_" in line for line in uses), uses
    load = next(line for line in uses if "__hip_atomic_load" in line)
    assert load.startswith("if (threadIdx.x == 0) state_s =")
    after = text[text.index(load) + len(load):].split(";")
    assert after[0].strip() == "__syncthreads()" and "bc_skip(state_s" in after[1]
    assert not re.search(r"bc_skip\(p\b", text)
