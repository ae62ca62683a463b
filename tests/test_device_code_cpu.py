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


def _registers(operand):
    """The vector registers that an operand names, as (file, number)."""
    out = []
    for kind, first, last, single in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", operand):
        out += [(kind, n) for n in range(int(first or single), int(last or single) + 1)]
    return out


@pytest.mark.skipif(OBJDUMP is None, reason="llvm-objdump not found")
def test_mfmas_keep_their_distance_from_vector_instructions(tmp_path):
    """An MFMA may read a register two wait states after a vector ALU instruction has written it, and other instructions may
    touch a 16x16 MFMA's result 8 (16-bit operands, K = 32) or 12 (e4m3, K = 128) wait states after its issue: what the
    compiler keeps between the ones that it knows.  The MFMAs that are written in inline assembly have to keep it by
    themselves."""
    import fuser_amd

    settle = {"v_mfma_f32_16x16x32": 8, "v_mfma_scale_f32_16x16x128": 12}
    mfmas, early = 0, []
    now, written, results = 0, {}, {}  # registers and when a vector ALU instruction wrote them / an MFMA's result may be used
    for name, operands in _instructions(Path(fuser_amd.__file__).parent / "libnvf_hip.so", tmp_path):
        if name == "s_nop":
            now += int(operands, 0) + 1
            continue
        now += 1
        if name in ("s_endpgm", "s_branch", "s_setpc_b64"):
            written.clear(), results.clear()
        elif "mfma" in name:
            parts = re.split(r",\s*(?![^\[]*\])", operands)
            mfmas += 1
            early += [f"{name} {operands}" for part in parts[1:] for r in _registers(part) if now - written.get(r, -9) <= 2]
            for prefix, states in settle.items():
                if name.startswith(prefix):
                    results.update({r: now + states for r in _registers(parts[0])})
        elif name.startswith(("v_", "ds_", "global_", "buffer_", "scratch_", "flat_")):
            if results:
                early += [f"{name} {operands}" for r in _registers(operands) if results.get(r, -9) >= now]
            if name.startswith("v_"):
                dest = operands if "swap" in name else re.split(r",\s*(?![^\[]*\])", operands)[0]
                written.update({r: now for r in _registers(dest)})
        if now % 64 == 0:
            results = {r: t for r, t in results.items() if t >= now}
    assert mfmas > 1000 and not early, f"{len(early)} instructions too early, e.g. {early[:3]}"
