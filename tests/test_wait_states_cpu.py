"""The machine code of the kernel library, as built here from its sources: a vector memory instruction reads no scalar register that
the vector ALU has written within the five instructions before it (the CDNA ISA documents list that as a wait the program has
to provide).  The compiler provides it for its own instructions, but not for the ones in inline assembly: the direct-to-LDS
loads with a scalar base."""
import os
import re
import struct
import subprocess

import pytest

from umdk_original_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
WAIT_STATES = 5


def _code_objects(path):
    """The gfx950 code objects in a library's offload bundles."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + name].decode()
            pos += 24 + name
            if "gfx950" in target:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


def _scalars(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"s(\d+)$", operand)
    return {int(m[1])} if m else set()


def _operands(text):
    return [w for part in text.split(None, 1)[1:] for t in part.split(",") for w in t.split()]


WRITES_SCALAR = re.compile(r"v_(readfirstlane|readlane|cmpx?_|add_co|sub_co|addc_co|subb_co|div_scale)")
NO_RESULT = re.compile(r"s_(waitcnt|nop|cbranch|branch|barrier|cmp|bitcmp|setprio|sleep|endpgm|sethalt)")


def _too_close(code):
    """Vector memory instructions that read a scalar register the vector ALU wrote fewer than WAIT_STATES before."""
    found = []
    for k, text in enumerate(code):
        if not re.match(r"(global|buffer|flat|scratch)_", text):
            continue
        want = set().union(*(_scalars(o) for o in _operands(text)), set())
        states, j = 0, k - 1
        while want and j >= 0 and states < WAIT_STATES:
            before = code[j]
            operands = _operands(before)
            if WRITES_SCALAR.match(before):
                # the result is the first operand, or the second of those that have a carry or a condition beside it
                if any(_scalars(o) & want for o in operands[:2] if not before.startswith("v_read") or o is operands[0]):
                    found.append(" ; ".join(code[j:k + 1]))
                    break
            elif before.startswith("s_") and not NO_RESULT.match(before) and operands:
                want -= _scalars(operands[0])   # what is read is the scalar ALU's, which needs no wait
            m = re.match(r"s_nop (\d+)", before)
            states += int(m[1]) + 1 if m else 1
            j -= 1
    return found


def test_the_check_sees_what_it_is_for():
    bad = ["v_readfirstlane_b32 s8, v78", "s_mov_b32 m0, s85", "s_nop 0", "global_load_lds_dword v76, s[8:9]"]
    assert _too_close(bad) == [" ; ".join(bad)]
    assert not _too_close(bad[:2] + ["s_nop 3"] + bad[3:])
    assert not _too_close(bad[:1] + ["s_add_u32 s8, s4, s6"] + bad[1:])
    assert _too_close(["v_cmp_eq_u32_e64 s[4:5], v0, v1", "buffer_load_dword v0, v1, s[4:7], 0 offen"])
    assert _too_close(["v_readlane_b32 s5, v255, 3", "global_store_dword v0, v1, s[4:5]"])
    assert not _too_close(["v_readlane_b32 s7, v255, s4", "global_store_dword v0, v1, s[4:5]"])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
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
