"""The machine code of the tile GEMM, as built here from its source.  Its K loop requests weights (FP8: and their scales) into
registers from inline assembly and waits for them by hand, and it names its accumulation registers itself; both rest on what the compiler makes of the code
around them:
  * from a request to the wait that covers it, no instruction on any path reads or writes the registers it loads into;
  * nothing but the multiplications, their clearing and the epilogue's reads touches an accumulation register, and nothing is
    spilled to memory."""
import re
import subprocess

from umdk_original_amd import build
from umdk_original_amd.machine_code import in_flight as _in_flight, kernels as _kernels
from test_wait_states_cpu import OBJDUMP, _code_objects


def test_the_check_sees_what_it_is_for():
    load = "buffer_load_dwordx4 v[4:7], v1, s[4:7], s8 offen"
    assert _in_flight([load, "v_mov_b32_e32 v9, v5", "s_waitcnt vmcnt(0)", "s_endpgm"], {})
    assert _in_flight([load, "buffer_load_dwordx4 v2, s[4:7], 0 offen lds", "s_waitcnt vmcnt(2)", "ds_read_b32 v6, v0", "s_endpgm"], {})
    assert not _in_flight([load, "buffer_load_dwordx4 v2, s[4:7], 0 offen lds", "s_waitcnt vmcnt(1)", "ds_read_b32 v6, v0", "s_endpgm"], {})
    # around a loop: the wait is in front of the use only on the way through the body
    loop = ["v_mov_b32_e32 v9, v5", "s_waitcnt vmcnt(0)", load, "s_cbranch_scc1 0", "s_waitcnt vmcnt(0)", "s_endpgm"]
    assert _in_flight(loop, {3: 0})
    assert not _in_flight([loop[1], loop[0]] + loop[2:], {3: 0})


def test_tile_gemm(tmp_path):
    kernels = 0
    for i, obj in enumerate(_code_objects(build.LIB_PATH)):
        f = tmp_path / ("%d.o" % i)
        f.write_bytes(obj)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], stdout=subprocess.PIPE, text=True, check=True).stdout
        if "11gemm_kernel" not in listing:
            continue
        for name, code, targets in _kernels(listing):
            if "11gemm_kernel" not in name:
                continue
            kernels += 1
            assert sum(t.startswith("v_mfma") for t in code) > 100
            for t in code:
                assert not t.startswith("scratch_"), t
                if re.search(r"\ba(\d+|\[)", t):
                    assert re.match(r"v_mfma_(i32_32x32x32_i8|scale_f32_32x32x64_f8f6f4) a\[|v_accvgpr_write_b32 a\d+, 0$|"
                                    r"v_accvgpr_read_b32 v\d+, a\d+$", t), t
            assert not _in_flight(code, targets)
    assert kernels == 2    # int8 and FP8
