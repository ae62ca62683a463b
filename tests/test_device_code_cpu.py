"""What the hand-written parts of the kernels owe the hardware, checked in the device code as it was built (no GPU needed)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:/opt/rocm/bin")


def _instructions(library, folder):
    """(name, operands) of every instruction of every gfx950 code object in the library, in the order of the code."""
    shutil.copy(library, folder)
    subprocess.run([OBJDUMP, "--offloading", library.name], cwd=folder, check=True, capture_output=True)
    objects = sorted(folder.glob("*gfx950"))
    assert objects
    for path in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", path.name], cwd=folder, check=True,
                              capture_output=True, text=True).stdout
        for line in text.splitlines():
            if line.startswith("\t"):
                name, _, operands = line.split("//")[0].strip().partition(" ")
                yield name, operands


@pytest.mark.skipif(OBJDUMP is None, reason="llvm-objdump not found")
def test_a_write_of_m0_is_a_wait_state_before_the_lds_direct_load_that_uses_it(tmp_path):
    """An LDS-direct load takes its LDS address from m0.  gfx9 needs one wait state after a scalar write of m0; the compiler
    inserts it for its own code, inside inline assembly it cannot."""
    import fuser_amd

    loads, early = 0, 0
    written = False  # by the instruction before
    for name, operands in _instructions(Path(fuser_amd.__file__).parent / "libnvf_hip.so", tmp_path):
        if re.match(r"(global|buffer|flat|scratch)_load", name) and ("_lds_" in name or operands.endswith(" lds")):
            loads += 1
            early += written
        written = name.startswith("s_") and operands.startswith("m0,")
    assert loads > 0 and early == 0, f"{early} of {loads} LDS-direct loads follow the write of m0 at once"
