"""Properties of the LM heads' kernels that only their assembly shows (CPU).

The GEMMs give padding rows no branch: their logits and tile words are stored
through a buffer resource that ends after the last real row, and the range
check drops them.  The check is certain only for the offset in the vector
register.  A store that carried the row in the scalar offset could, with fewer
rows than that offset reaches over, write past the caller's buffer.

The narrow GEMM's block loop requests its operands two blocks ahead.  If the
compiler moves a loaded register at the loop's edge, it waits there for every
load in flight, and each round then pays a memory round trip.
"""
import pathlib
import re
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "promptboot_amd" / "csrc"


def make_variable(name: str) -> str:
    """The value that the Makefile builds the library with."""
    out = subprocess.run(["make", "-s", "-C", str(CSRC), "--eval", f"print:; @echo '$({name})'", "print"],
                         check=True, capture_output=True, text=True)
    return out.stdout.strip()


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: its assembly lines} of the head's GEMMs."""
    hipcc = make_variable("HIPCC")
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    asm = tmp_path_factory.mktemp("asm") / "lmhead.s"
    subprocess.run([hipcc, *make_variable("HIPFLAGS").split(), "-w", "--cuda-device-only", "-S", "-o", str(asm),
                    str(CSRC / "pb_lmhead.hip")], check=True, capture_output=True)
    found, lines = {}, None
    for line in asm.read_text().splitlines():
        label = re.match(r"(_Z\w+):", line)
        if label:
            lines = found.setdefault(label.group(1), []) if "lm_gemm" in label.group(1) else None
        elif line.startswith(".Lfunc_end"):
            lines = None
        elif lines is not None:
            lines.append(line.split(";")[0].strip())
    return found


def test_no_buffer_store_of_the_heads_has_a_scalar_offset(kernels):
    stores, bad = 0, []
    for name, lines in kernels.items():
        for line in lines:
            # buffer_store_dwordx2 v[0:1], v2, s[4:7], 0 offen nt
            store = re.match(r"buffer_store_\w+ \S+, (?:\S+, )?s\[\d+:\d+\], (\S+)", line)
            if store:
                stores += 1
                if store.group(1) != "0":
                    bad.append((name, line))
    assert stores > 100, stores  # the pattern still finds them
    assert not bad, (len(bad), bad[:4])


# row groups, result registers, fused quantisation: 1, 2, 3-4, 17-24, 25-32, 33-48 and 49-64 rows
@pytest.mark.parametrize("groups, regs, fused", [(1, 1, 1), (1, 2, 1), (1, 4, 1), (1, 12, 0), (1, 16, 0),
                                                 (2, 12, 0), (2, 16, 0)])
def test_the_narrow_q4_0_loop_keeps_its_loads_in_flight(kernels, groups, regs, fused):
    name = f"lm_gemm_narrow_kernelILb0ELi{groups}ELi{regs}ELb{fused}ELi4EE"
    lines = next(v for k, v in kernels.items() if name in k)
    starts = {line[:-1]: i for i, line in enumerate(lines) if re.fullmatch(r"\.LBB\w+:", line)}
    loops = []
    for i, line in enumerate(lines):
        back = re.fullmatch(r"s_cbranch_\w+ (\.LBB\w+)", line)
        if back and starts[back.group(1)] < i:
            body = lines[starts[back.group(1)]:i]
            if sum("v_mfma_i32_32x32x32" in x for x in body) == 4:  # two blocks, two column tiles each
                loops.append(body)
    assert len(loops) == 1
    waits = [int(m.group(1)) for line in loops[0] if (m := re.search(r"vmcnt\((\d+)\)", line))]
    assert waits and min(waits) > 0, waits
