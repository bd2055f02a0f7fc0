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


FMAC = "v_fmac_f64_dpp v[0:1], v[2:3], v[4:5] row_newbcast:1 row_mask:0xf bank_mask:0xf"


@pytest.mark.parametrize("lines,bad", [
    (["v_add_f64 v[2:3], v[6:7], v[8:9]", FMAC], 1),
    (["v_add_f64 v[2:3], v[6:7], v[8:9]", "s_nop 0", FMAC], 1),
    (["v_add_f64 v[2:3], v[6:7], v[8:9]", "s_nop 1", FMAC], 0),
    (["v_mov_b32_e32 v3, v8", "v_mul_f64 v[6:7], v[8:9], v[8:9]", FMAC], 1),
    (["v_accvgpr_read_b32 v2, a8", FMAC], 1),
    (["v_add_f64 v[4:5], v[6:7], v[8:9]", FMAC], 0),       # (the other sources are not read from other lanes)
    (["v_add_f64 v[0:1], v[6:7], v[8:9]", FMAC], 0),
    (["v_rcp_f64_e32 v[4:5], v[6:7]", FMAC], 1),
    (["v_rcp_f64_e32 v[4:5], v[6:7]", "s_nop 0", FMAC], 0),
    (["v_cmpx_lt_f64_e32 v[6:7], v[8:9]", "s_nop 3", FMAC], 1),
    (["v_cmpx_lt_f64_e32 v[6:7], v[8:9]", "s_nop 4", FMAC], 0),
    (["ds_read_b64 v[2:3], v9", "s_waitcnt lgkmcnt(0)", FMAC], 0),
    (["v_permlane32_swap_b32_e32 v7, v3", FMAC], 1),
    # written at the end of a loop whose head uses it
    (["s_nop 1", FMAC, "v_mov_b32_e32 v2, v8", "s_cbranch_scc1 1", "s_endpgm"], 1),
    (["s_nop 1", FMAC, "v_mov_b32_e32 v2, v8", "s_cbranch_scc1 0", "s_endpgm"], 0),
    (["s_nop 0", "v_mov_b32_e32 v2, v8", "s_branch 5", FMAC, "s_nop 0", "s_nop 1", FMAC], 0),
])
def test_sources_from_other_lanes(lines, bad):
    (kernel,) = check.kernels(_listing(lines))
    found, looked_at = check.violations(kernel)
    assert looked_at == sum("_dpp" in t for t in lines)
    assert len(found) == bad


def test_built_library_keeps_its_wait_states():
    library = os.path.join(os.path.dirname(CSRC), "libsymmetrix_amd.so")
    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(library) or not os.path.exists(objdump):
        pytest.skip("no built library or no llvm-objdump here")
    found, looked_at = check.check(library, objdump)
    assert looked_at > 0
    assert not found, found[:5]
