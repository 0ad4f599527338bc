"""Properties of the device code that a run on the GPU cannot show, checked on
its source and on the listing of the built library (no GPU calls)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from mak_mi355x import _build, _lib

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


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """The instructions of every kernel of the built library, in order."""
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not Path(objdump).exists():
        pytest.skip("no llvm-objdump")
    _lib.load()
    where = tmp_path_factory.mktemp("listing")
    shutil.copy(_build.LIB, where / "lib.so")
    subprocess.run([objdump, "--offloading", "lib.so"], cwd=where, check=True, capture_output=True)
    out = []
    for f in sorted(where.glob(f"*{_build.ARCH}")):
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", f.name], cwd=where, check=True,
                              capture_output=True, text=True).stdout
        out += [line.split("//")[0].strip() for line in text.splitlines()]
    return out


@pytest.fixture(scope="module")
def listing_by_kernel(listing):
    """The set of opcodes of each kernel, by its mangled name."""
    out, name = {}, None
    for line in listing:
        head = re.fullmatch(r"[0-9a-f]+ <(\S+)>:", line)
        if head:
            name = head[1]
            out.setdefault(name, set())
        elif name is not None and line:
            out[name].add(line.split()[0])
    return out


def registers(operand):
    """The VGPR numbers of an operand such as v7, -v[4:5]."""
    m = re.fullmatch(r"-?\|?v(?:(\d+)|\[(\d+):(\d+)\])\|?", operand.strip())
    if m is None:
        return set()
    return {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))


def test_dpp_sources_are_waited_for(listing):
    """A VGPR may be the source of a DPP read from two wait states after the
    VALU instruction that wrote it.  The compiler keeps that for its own
    instructions and cannot see into an asm block, so (1) no DPP read of the
    library is closer than that to its source's write, and (2) the multiply-adds
    that only asm blocks contain follow a wait of their block, or two products
    in its place, without any other instruction between, so that (1) does not
    rest on where the register allocator puts its copies."""
    recent, led, before = [], False, ""      # (registers written, wait states) of the last instructions
    reads = blocks = 0
    close, loose = [], []
    for line in listing:
        if not line or line.endswith(":"):
            recent, led, before = [], False, ""
            continue
        op, _, rest = line.partition(" ")
        operands = re.split(r",\s*(?![^\[]*\])", rest.split(" row_")[0])
        if "_dpp" in op:
            reads += 1
            source, states = registers(operands[1]), 0
            for written, n in reversed(recent):
                if states >= 2:
                    break
                if written & source:
                    close.append(line)
                states += n
            if op.startswith("v_fmac_f64_dpp"):
                blocks += 1
                if not led:
                    loose.append(line)
        led = ((op == "s_nop" and int(rest) >= 1) or op == before == "v_mul_f64"
               or (led and op.startswith("v_fmac_f64_dpp")))
        before = op
        wrote = registers(operands[0]) if op.startswith("v_") else set()
        recent = recent[-7:] + [(wrote, int(rest) + 1 if op == "s_nop" else 1)]
    assert reads > 1000 and blocks > 1000, (reads, blocks)
    assert not close, (len(close), close[:3])
    assert not loose, (len(loose), loose[:3])


def test_batched_blocks_stay_in_64_bits(listing_by_kernel):
    """The batched factorisation of whole blocks is Float64 / ComplexF64
    throughout: no kernel of it converts to 32 bits or multiplies in them."""
    kernels = {k: v for k, v in listing_by_kernel.items() if "bchol" in k or "qr_small" in k or "qr_tall" in k}
    assert len(kernels) >= 15, sorted(kernels)
    for name, ops in kernels.items():
        low = {op for op in ops if re.match(r"v_mfma_f32|v_cvt_f32_f64|v_cvt_f16|v_cvt_pk_bf16|v_fma(c|mk|ak)?_f32", op)}
        assert not low, (name, low)
