"""The machine code of the kernel library, as built here from its sources: a vector memory instruction reads no scalar register that
the vector ALU has written within the five instructions before it (the CDNA ISA documents list that as a wait the program has
to provide).  The compiler provides it for its own instructions, but not for the ones in inline assembly: the direct-to-LDS
loads with a scalar base."""
import subprocess

from umdk_original_amd import build
from umdk_original_amd.machine_code import OBJDUMP, code_objects as _code_objects, too_close as _too_close


def test_the_check_sees_what_it_is_for():
    bad = ["v_readfirstlane_b32 s8, v78", "s_mov_b32 m0, s85", "s_nop 0", "global_load_lds_dword v76, s[8:9]"]
    assert _too_close(bad) == [" ; ".join(bad)]
    assert not _too_close(bad[:2] + ["s_nop 3"] + bad[3:])
    assert not _too_close(bad[:1] + ["s_add_u32 s8, s4, s6"] + bad[1:])
    assert _too_close(["v_cmp_eq_u32_e64 s[4:5], v0, v1", "buffer_load_dword v0, v1, s[4:7], 0 offen"])
    assert _too_close(["v_readlane_b32 s5, v255, 3", "global_store_dword v0, v1, s[4:5]"])
    assert not _too_close(["v_readlane_b32 s7, v255, s4", "global_store_dword v0, v1, s[4:5]"])


def test_no_load_reads_a_scalar_too_soon(tmp_path):
    objects = list(_code_objects(build.LIB_PATH))
    assert len(objects) >= 5    # plan, dispatch, combine, and the two GEMMs
    loads = 0
    for i, obj in enumerate(objects):
        f = tmp_path / ("%d.o" % i)
        f.write_bytes(obj)
        p = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], stdout=subprocess.PIPE, text=True, check=True)
        code = [line.split("//")[0].strip() for line in p.stdout.splitlines() if line.startswith("\t")]
        loads += sum("global_load_lds" in text for text in code)
        assert not _too_close(code)
    assert loads > 100          # the direct-to-LDS loads of both GEMMs are among them
