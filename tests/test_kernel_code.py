"""The gfx950 code of the GEMM kernels, disassembled from the built
``libmxgg.so`` (no GPU needed).

The kernels issue their global -> LDS copies in inline asm and depend on
register behaviour the compiler does not model, so what matters is the code
that came out of it.
"""

import os
import re
import subprocess

import pytest

from test_kernel_resources import LIB, _code_objects

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """{kernel symbol: instructions, operands included} of the GEMM kernels."""
    if not os.path.exists(LIB):
        pytest.skip("libmxgg.so is not built (run __graft_entry__.build())")
    if not os.path.exists(OBJDUMP):
        pytest.skip("llvm-objdump not found")
    out = {}
    for i, co in enumerate(_code_objects(open(LIB, "rb").read())):
        p = tmp_path_factory.mktemp("code") / f"{i}.co"
        p.write_bytes(co)
        asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(p)], capture_output=True,
                             text=True, check=True).stdout
        for name, body in re.findall(r"^<(\w+)>:\n(.*?)(?=\n\n|\Z)", asm, re.S | re.M):
            if re.search(r"(fwd|wgrad|fwd_quad|fwd_stream)_kernel", name):
                out[name] = [ln.split("//")[0].split() for ln in body.splitlines() if ln.strip()]
    assert out
    return out


def _regs(operand, kind):
    """Register numbers of operand "v7" / "s[4:7]" of the given kind."""
    m = re.match(kind + r"(?:(\d+)|\[(\d+):(\d+)\])$", operand.strip(","))
    if not m:
        return set()
    return {int(m.group(1))} if m.group(1) else set(range(int(m.group(2)), int(m.group(3)) + 1))


def _idle(ins):
    """Issue slots an instruction takes."""
    return int(ins[1]) + 1 if ins[0] == "s_nop" else 1


def test_mfma_scales_are_not_overwritten_at_once(code):
    """The compiler does not guard the scale operands of v_mfma_scale_* as
    reads in flight: no vector instruction may write them in the four issue
    slots after it."""
    seen, bad = 0, []
    for name, ins in code.items():
        for i, x in enumerate(ins):
            if not x[0].startswith("v_mfma_scale"):
                continue
            seen += 1
            scales = _regs(x[5], "v") | _regs(x[6], "v")
            slots, k = 0, i + 1
            while slots < 4 and k < len(ins) and not ins[k][0].startswith(("s_branch", "s_cbranch")):
                op = ins[k][0]
                writes = _regs(ins[k][1], "v") if op.startswith(("v_", "ds_read")) and not op.startswith("v_mfma") else set()
                if writes & scales:
                    bad.append((name, " ".join(x), " ".join(ins[k]), slots))
                slots += _idle(ins[k])
                k += 1
    assert seen and not bad, bad[:5]


def test_accumulators_are_cleared_and_read_once(code):
    """Every accumulator of a 256 x 256 tile is cleared once (the weight
    gradient: once more for an empty group) and read once by the epilogue,
    with no moves between: at 4 cycles each they cost a tile up to 1.4 us."""
    seen = 0
    for name, ins in code.items():
        if "_kernelINS_3CfgILi256ELi256E" not in name or "fwd_quad" in name:
            continue
        seen += 1
        moves = sum(x[0].startswith("v_accvgpr") for x in ins)
        assert moves <= (3 if "wgrad" in name else 2) * 256 + 16, (name, moves)
    assert seen


def test_lds_copies_find_their_scalar_operands(code):
    """The hardware needs five wait states between a vector instruction that
    writes a scalar register and a copy that reads it, and one between a write
    of M0 and an LDS copy; the compiler adds none around asm.  M0 is written
    for the copies only."""
    seen, bad = 0, []
    for name, ins in code.items():
        for i, x in enumerate(ins):
            if x[0].startswith(("s_", "v_readfirstlane")) and len(x) > 1 and x[1] == "m0,":
                if ins[i + 1][0] != "s_nop":
                    bad.append((name, " ".join(x), " ".join(ins[i + 1])))
            if not (x[0].startswith("buffer_load") and "lds" in x[-1]):
                continue
            seen += 1
            reads = set().union(*(_regs(t, "s") for t in x[1:]))
            slots, k = 0, i - 1
            while slots < 5 and k >= 0:
                if ins[k][0].startswith("v_") and len(ins[k]) > 1 and _regs(ins[k][1], "s") & reads:
                    bad.append((name, " ".join(ins[k]), " ".join(x), slots))
                slots += _idle(ins[k])
                k -= 1
    assert seen and not bad, bad[:5]
