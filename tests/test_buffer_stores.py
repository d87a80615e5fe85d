"""The LM heads' buffer stores, read from the assembly of the kernels (CPU).

The GEMMs give padding rows no branch: their logits and tile words are stored
through a buffer resource that ends after the last real row, and the range
check drops them.  The check is certain only for the offset in the vector
register.  A store that carried the row in the scalar offset could, with fewer
rows than that offset reaches over, write past the caller's buffer.
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


def test_no_buffer_store_of_the_heads_has_a_scalar_offset(tmp_path):
    hipcc = make_variable("HIPCC")
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    asm = tmp_path / "lmhead.s"
    subprocess.run([hipcc, *make_variable("HIPFLAGS").split(), "-w", "--cuda-device-only", "-S", "-o", str(asm),
                    str(CSRC / "pb_lmhead.hip")], check=True, capture_output=True)
    stores = 0
    bad = []
    kernel = None
    for line in asm.read_text().splitlines():
        label = re.match(r"(_Z\w+):", line)
        if label:
            kernel = label.group(1)
        # buffer_store_dwordx2 v[0:1], v2, s[4:7], 0 offen nt
        store = re.match(r"\s+buffer_store_\w+ \S+, (?:\S+, )?s\[\d+:\d+\], (\S+)", line)
        if store and kernel and "lm_gemm" in kernel:
            stores += 1
            if store.group(1) != "0":
                bad.append((kernel, line.strip()))
    assert stores > 100, stores  # the pattern still finds them
    assert not bad, (len(bad), bad[:4])
