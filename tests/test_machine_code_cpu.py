"""What build.py looks for in the machine code of the kernel library, and that it does: on listings with a fault written into them,
and on the library as built.  (The older checks have files of their own: test_wait_states_cpu.py,
test_registers_in_flight_cpu.py.)"""
import os

import pytest

from umdk_original_amd import build, machine_code

MULTIPLY = "v_mfma_i32_32x32x32_i8 a[0:15], v[4:7], v[8:11], a[0:15]"


@pytest.mark.parametrize("before", ["v_mov_b32_e32 v9, v1", "v_accvgpr_write_b32 a15, 0", "v_lshl_add_u64 v[6:7], v[0:1], 3, v[2:3]",
                                    "v_swap_b32 v1, v4"])
def test_operands_of_a_multiplication(before):
    look = machine_code.operands_too_close
    assert look([before, MULTIPLY], {}) == look([before, "s_nop 0", MULTIPLY], {}) == ["%s ... %s" % (before, MULTIPLY)]
    assert not look([before, "s_nop 1", MULTIPLY], {})
    assert not look([before, "v_mov_b32_e32 v20, v1", "ds_read_b32 v21, v1", MULTIPLY], {})
    # around a loop: in front of the multiplication only on the way back
    loop = [MULTIPLY, "s_nop 4", before, "s_cbranch_scc1 0", "s_endpgm"]
    assert look(loop, {3: 0}) and not look(loop, {})
    assert not look(["s_nop 4", before, "s_branch 0", MULTIPLY], {2: 0})    # nothing falls through from a branch


def test_a_scalar_on_the_way_back_of_a_loop():
    loop = ["global_load_dword v0, v1, s[8:9]", "s_nop 4", "v_readfirstlane_b32 s8, v78", "s_cbranch_scc1 0", "s_endpgm"]
    assert machine_code.too_close(loop, {3: 0}) and not machine_code.too_close(loop, {})
    assert not machine_code.too_close(loop[:3] + ["s_nop 3"] + loop[3:], {4: 0})
    assert not machine_code.too_close(loop[:3] + ["s_mov_b32 s8, s4"] + loop[3:], {4: 0})


def test_what_is_no_operand():
    for other in ("v_cmp_eq_u32_e32 vcc, v4, v5", "v_readfirstlane_b32 s8, v4", "v_mov_b32_e32 v20, v4", MULTIPLY):
        assert not machine_code.operands_too_close([other, MULTIPLY], {})


def _listing(name, code):
    return "0000000000001000 <%s>:\n" % name + "".join("\t%s // %012X:\n" % (t, 0x1000 + 8 * i) for i, t in enumerate(code))


GOOD = ["buffer_load_dwordx4 v[20:23], v1, s[4:7], s8 offen", "s_waitcnt vmcnt(0)", "v_mov_b32_e32 v0, v20"] + [MULTIPLY] * 101
TILE = "_ZN3cam12_GLOBAL__N_111gemm_kernelILb%dEEEvNS_8GemmArgsE"


@pytest.mark.parametrize("fault", [
    (0, "v_readlane_b32 s8, v1, 3"),            # in front of the load that reads it
    (1, "v_mov_b32_e32 v0, v21"),               # of a register under way
    (3, "v_mov_b32_e32 v4, v20"),               # in front of the first multiplication
    (3, "v_accvgpr_write_b32 a40, v20"),        # a value parked in an accumulation register
    (3, "scratch_store_dword off, v20, s32"),
    (3, "s_swappc_b64 s[30:31], s[16:17]")])
def test_the_build_gives_no_such_library(monkeypatch, tmp_path, fault):
    class Done:
        returncode = 0

        def __init__(self, cmd, **_):
            open(cmd[cmd.index("-o") + 1], "w").close()

        def communicate(self):
            return "", None

    at, text = fault
    bad = GOOD[:at] + [text] + GOOD[at:]
    code = {"good": [GOOD, GOOD], "bad": [GOOD, bad]}
    library = tmp_path / "library.so"
    monkeypatch.setattr(build, "LIB_DIR", str(tmp_path))
    monkeypatch.setattr(build, "LIB_PATH", str(library))
    monkeypatch.setattr(build.subprocess, "Popen", Done)
    monkeypatch.setattr(build.subprocess, "check_call", Done)
    for part in ("build_calib", "build_abi_consumer", "build_torch_libraries"):
        monkeypatch.setattr(build, part, lambda verbose: None)
    for kind in ("good", "bad"):
        monkeypatch.setattr(machine_code, "listings", lambda path: [_listing(TILE % i, c) for i, c in enumerate(code[kind])])
        if kind == "good":
            assert build.build() == str(library) and library.exists()
        else:
            with pytest.raises(RuntimeError, match="machine code"):
                build.build()
            assert not library.exists()
    monkeypatch.setattr(machine_code, "listings", lambda path: [])   # nothing was looked at
    with pytest.raises(RuntimeError, match="0 kernels"):
        build.build()


def test_the_library_as_built():
    assert os.path.exists(build.LIB_PATH)
    assert machine_code.faults(build.LIB_PATH) == []


@pytest.mark.parametrize("plainly", [False, True])
def test_how_quantised_tokens_are_stored(plainly):
    """What the plan's first launch leaves for a GEMM that gathers: tiles of few rows are slower behind plain stores."""
    found = [[t for t in code if t.startswith("global_store_dwordx2")] for listing in machine_code.listings(build.LIB_PATH)
             for name, code, _ in machine_code.kernels(listing) if "plan_quant_kernel" in name and "Lb%dEEE" % plainly in name]
    assert len(found) == 6 and all(len(stores) >= 8 and all(t.endswith(" nt") != plainly for t in stores) for stores in found)
