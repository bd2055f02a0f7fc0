"""The check of the built device code (wait states around inline assembly): on listings written here, and on the library."""
import os
import sys

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "symmetrix_amd", "csrc")
sys.path.insert(0, CSRC)
import check_device_code as check  # noqa: E402


def _listing(lines):
    """A function at 0x1000, four bytes an instruction; a branch names the line it goes to."""
    out = ["", "0000000000001000 <f>:"]
    for i, text in enumerate(lines):
        mnemonic, _, operands = text.partition(" ")
        tail = ""
        if "branch" in mnemonic:
            tail = f" <f+0x{4 * int(operands):x}>"
        out.append(f"\t{mnemonic} {operands}    // {0x1000 + 4 * i:012X}: 00000000{tail}")
    return "\n".join(out)


LOAD = "global_load_lds_dwordx4 v[4:5], off"


@pytest.mark.parametrize("lines,bad", [
    (["s_mov_b32 m0, s4", LOAD, "s_endpgm"], 1),
    (["s_mov_b32 m0, s4", "s_nop 0", LOAD, "s_endpgm"], 0),
    (["s_add_i32 m0, s2, 4", "v_mov_b32_e32 v1, 0", LOAD, "s_endpgm"], 0),
    (["s_mov_b32 s4, m0", LOAD, "s_endpgm"], 0),
    # the write is right before the load on the way round a loop only
    (["s_mov_b32 m0, s4", "s_nop 0", LOAD, "s_mov_b32 m0, s5", "s_cbranch_scc1 2", "s_endpgm"], 0),
    (["s_mov_b32 m0, s4", "s_branch 3", "s_endpgm", LOAD, "s_endpgm"], 0),
    (["s_nop 0", LOAD, "s_endpgm", "s_mov_b32 m0, s5", LOAD], 1),
])
def test_lds_loads_and_m0(lines, bad):
    (kernel,) = check.kernels(_listing(lines))
    found, looked_at = check.violations(kernel)
    assert looked_at == sum("load_lds" in t for t in lines)
    assert len(found) == bad


def test_built_library_keeps_its_wait_states():
    library = os.path.join(os.path.dirname(CSRC), "libsymmetrix_amd.so")
    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(library) or not os.path.exists(objdump):
        pytest.skip("no built library or no llvm-objdump here")
    found, looked_at = check.check(library, objdump)
    assert looked_at > 0
    assert not found, found[:5]
