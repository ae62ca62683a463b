"""What the hand-written parts of the kernels owe the hardware, checked in the device code as it was built (no GPU needed)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:/opt/rocm/bin")


def _code(library, folder):
    """The gfx950 code objects in the library: for each a list of (address, name, operands) in the order of the code."""
    shutil.copy(library, folder)
    subprocess.run([OBJDUMP, "--offloading", library.name], cwd=folder, check=True, capture_output=True)
    objects = sorted(folder.glob("*gfx950"))
    assert objects
    for path in objects:
        text = subprocess.run([OBJDUMP, "-d", path.name], cwd=folder, check=True, capture_output=True, text=True).stdout
        code = []
        for line in text.splitlines():
            instruction, _, encoding = line.partition("//")
            if line.startswith("\t") and encoding:
                name, _, operands = instruction.strip().partition(" ")
                code.append((int(encoding.split(":")[0], 16), name, operands.strip()))
        yield code


def _instructions(library, folder):
    """(name, operands) of every instruction of every gfx950 code object in the library, in the order of the code."""
    for code in _code(library, folder):
        for _, name, operands in code:
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


def _operands(operands):
    return re.split(r",\s*(?![^\[]*\])", operands)


def _followers(code, at, index, states):
    """(index, wait states in between) of the instructions that are reached from instruction `index` with fewer than `states`
    wait states in between, over every branch both ways: the way from a loop's end back to its beginning is one of them."""
    todo, seen = [(index, -1)], {}
    while todo:
        i, between = todo.pop()
        address, name, operands = code[i]
        here = between + (int(operands, 0) + 1 if name == "s_nop" else 1)
        if here >= states or name in ("s_endpgm", "s_setpc_b64"):
            continue
        following = [i + 1] if name != "s_branch" else []
        if name.startswith(("s_branch", "s_cbranch")):
            offset = int(operands.split()[0], 0)
            following.append(at[address + 4 + 4 * (offset - 65536 if offset > 32767 else offset)])
        for j in following:
            if j < len(code) and seen.get(j, states) > here:
                seen[j] = here
                todo.append((j, here))
    return seen.items()


def _too_early(code):
    """Number of MFMAs, and the instructions that come too few wait states after one that they depend on."""
    settle = {"v_mfma_f32_16x16x32": (8, 7), "v_mfma_scale_f32_16x16x128": (12, 12)}  # before the result is read, before it is written
    at = {address: i for i, (address, _, _) in enumerate(code)}
    mfma = [("mfma" in name) for _, name, _ in code]
    branch = [name.startswith(("s_branch", "s_cbranch")) for _, name, _ in code]
    early = []
    for i, (_, name, operands) in enumerate(code):
        if mfma[i]:
            read, write = next((n for prefix, n in settle.items() if name.startswith(prefix)), (0, 0))
            result = set(_registers(_operands(operands)[0])) if read else ()
            for j, between in _followers(code, at, i, read):
                if not mfma[j] and code[j][1].startswith(("v_", "ds_", "global_", "buffer_", "scratch_", "flat_")):
                    parts = _operands(code[j][2])
                    if between >= write and code[j][1].startswith("v_") and "swap" not in code[j][1]:
                        parts = parts[1:]  # (the first one is written)
                    if result & {r for part in parts for r in _registers(part)}:
                        early.append(f"{code[j][1]} {code[j][2]} after {name}")
        elif name.startswith("v_") and any(mfma[i + 1 : i + 3]) | any(branch[i + 1 : i + 3]):
            for j, between in _followers(code, at, i, 2):
                if mfma[j]:
                    written = set(_registers(operands if "swap" in name else _operands(operands)[0]))
                    if written & {r for part in _operands(code[j][2])[1:] for r in _registers(part)}:
                        early.append(f"{code[j][1]} {code[j][2]} after {name}")
    return sum(mfma), early


@pytest.mark.skipif(OBJDUMP is None, reason="llvm-objdump not found")
def test_mfmas_keep_their_distance_from_vector_instructions(tmp_path):
    """An MFMA may read a register two wait states after a vector ALU instruction has written it, and other instructions may
    read a 16x16 MFMA's result 8 (16-bit operands, K = 32) or 12 (e4m3, K = 128) wait states after its issue, and overwrite it
    7 or 12 states after: what the compiler keeps between the ones that it knows.  The MFMAs that are written in inline assembly have to keep it by
    themselves, along every path: from the end of a loop to its beginning too."""
    import fuser_amd

    found = [_too_early(code) for code in _code(Path(fuser_amd.__file__).parent / "libnvf_hip.so", tmp_path)]
    early = [e for _, es in found for e in es]
    assert sum(mfmas for mfmas, _ in found) > 1000 and not early, f"{len(early)} instructions too early, e.g. {early[:3]}"


def test_the_distance_is_taken_over_branches_too():
    """A loop whose last instruction writes what its first MFMA reads, and an MFMA whose result is read past a forward branch."""
    mfma = "v_mfma_f32_16x16x32_f16"
    loop = [(0, mfma, "a[0:3], v[0:3], v[4:7], a[0:3]"), (8, "s_nop", "7"), (12, "v_mov_b32_e32", "v5, v9"), (16, "s_cbranch_scc1", "65531"), (20, "s_endpgm", "")]
    assert _too_early(loop) == (1, [f"{mfma} a[0:3], v[0:3], v[4:7], a[0:3] after v_mov_b32_e32"])
    assert _too_early([*loop[:2], (12, "v_mov_b32_e32", "v5, v9"), (16, "s_nop", "0"), (20, "s_cbranch_scc1", "65530"), loop[4]])[1] == []
    read = [(0, mfma, "a[0:3], v[0:3], v[4:7], a[0:3]"), (8, "s_branch", "2"), (12, "s_nop", "15"), (16, "s_endpgm", ""), (20, "v_accvgpr_read_b32", "v1, a2"), (24, "s_endpgm", "")]
    assert _too_early(read)[1] == [f"v_accvgpr_read_b32 v1, a2 after {mfma}"]
    assert _too_early([*read[:1], (8, "s_nop", "6"), (12, "s_branch", "2"), *[(a + 4, n, o) for a, n, o in read[2:]]])[1] == []
