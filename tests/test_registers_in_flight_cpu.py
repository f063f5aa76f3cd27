"""The machine code of the tile GEMM, as built here from its source.  Its K loop requests weights (FP8: and their scales) into
registers from inline assembly and waits for them by hand, and it names its accumulation registers itself; both rest on what the compiler makes of the code
around them:
  * from a request to the wait that covers it, no instruction on any path reads or writes the registers it loads into;
  * nothing but the multiplications, their clearing and the epilogue's reads touches an accumulation register, and nothing is
    spilled to memory."""
import os
import re
import subprocess

import pytest

from umdk_original_amd import build
from test_wait_states_cpu import OBJDUMP, _code_objects

VMEM = re.compile(r"(buffer|global|flat|scratch)_")


def _registers(text):
    found = set()
    for lo, hi in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        found.update(range(int(lo), int(hi) + 1))
    found.update(int(r) for r in re.findall(r"\bv(\d+)\b", text))
    return found


def _in_flight(code, targets):
    """Instructions that touch the registers of a load (to registers, not to LDS) which may still be under way."""
    touched = [_registers(text) for text in code]
    waits = [int(m[1]) if (m := re.search(r"vmcnt\((\d+)\)", t)) and t.startswith("s_waitcnt") else None for t in code]
    found = []
    for start, text in enumerate(code):
        if not re.match(r"(buffer|global)_load_\w+ v", text) or "_lds_" in text or text.endswith("lds"):
            continue
        dst = _registers(text.split(",")[0])
        todo, seen = [(start + 1, 0)], set()
        while todo:
            at, younger = todo.pop()
            while at < len(code) and (at, younger) not in seen:
                seen.add((at, younger))
                if waits[at] is not None and waits[at] <= younger:
                    break                        # loads retire in order: this one has come
                if touched[at] & dst:
                    found.append("%s ... %s" % (text, code[at]))
                    break
                if VMEM.match(code[at]):
                    younger += 1
                if code[at].startswith(("s_endpgm", "s_setpc")):
                    break
                if at in targets:
                    if code[at].startswith("s_branch"):
                        at = targets[at]
                        continue
                    todo.append((targets[at], younger))
                at += 1
    return found


def _kernels(listing):
    """name -> instructions and branch targets (by index) of every function in a disassembly."""
    name, base, rows = None, {}, {}
    for line in listing.splitlines():
        m = re.match(r"([0-9a-f]+) <(.+)>:", line)
        if m:
            name = m[2]
            base[name], rows[name] = int(m[1], 16), []
        elif name and line.startswith("\t") and "//" in line:
            text, note = (line.split("//") + [""])[:2]
            addr = int(note.split(":")[0], 16)
            jump = re.search(r"<%s\+0x([0-9a-f]+)>" % re.escape(name), note) if text.strip().startswith(("s_cbranch", "s_branch")) else None
            rows[name].append((addr, text.strip(), base[name] + int(jump[1], 16) if jump else None))
    for name, r in rows.items():
        index = {addr: i for i, (addr, _, _) in enumerate(r)}
        yield name, [t for _, t, _ in r], {i: index[to] for i, (_, _, to) in enumerate(r) if to is not None}


def test_the_check_sees_what_it_is_for():
    load = "buffer_load_dwordx4 v[4:7], v1, s[4:7], s8 offen"
    assert _in_flight([load, "v_mov_b32_e32 v9, v5", "s_waitcnt vmcnt(0)", "s_endpgm"], {})
    assert _in_flight([load, "buffer_load_dwordx4 v2, s[4:7], 0 offen lds", "s_waitcnt vmcnt(2)", "ds_read_b32 v6, v0", "s_endpgm"], {})
    assert not _in_flight([load, "buffer_load_dwordx4 v2, s[4:7], 0 offen lds", "s_waitcnt vmcnt(1)", "ds_read_b32 v6, v0", "s_endpgm"], {})
    # around a loop: the wait is in front of the use only on the way through the body
    loop = ["v_mov_b32_e32 v9, v5", "s_waitcnt vmcnt(0)", load, "s_cbranch_scc1 0", "s_waitcnt vmcnt(0)", "s_endpgm"]
    assert _in_flight(loop, {3: 0})
    assert not _in_flight([loop[1], loop[0]] + loop[2:], {3: 0})


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
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
