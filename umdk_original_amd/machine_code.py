"""Looks over the machine code of the kernel library after it has been built from its sources.

The kernels issue loads and multiplications from inline assembly, wait for them by hand and name the accumulation registers
themselves.  That is sound only for what the compiler made of the code around: it does not know that a register is being
loaded into, provides no wait states for instructions in inline assembly, and is free to copy, spill or move values there.
build.py runs check() on every library that it links, so that a compiler, a flag or a change of the source for which it does
not hold gives no library instead of one with wrong results now and then:
  * a vector memory instruction reads no scalar register that the vector ALU has written within the five wait states before
    it (the CDNA ISA documents list that as a wait the program has to provide);
  * a multiplication reads no register that the vector ALU has written within the two wait states before it (what the
    compiler keeps where the multiplications are its own instructions);
  * from a load into registers to the wait that covers it, no instruction on any path reads or writes these registers;
  * in the tile GEMM nothing but the multiplications, their clearing and the epilogue's reads touches an accumulation
    register, nothing is spilled to memory, and there is no call, which the walk along the paths would not follow."""
import os
import re
import struct
import subprocess
import tempfile

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
WAIT_STATES = 5            # from the vector ALU's write of a scalar register to a vector memory instruction that reads it
OPERAND_WAIT_STATES = 2    # from its write of a vector (accumulation) register to a multiplication that reads it
TILE_GEMM = "11gemm_kernel"   # in the mangled names of the tile GEMM's two kernels

VMEM = re.compile(r"(buffer|global|flat|scratch)_")
WRITES_SCALAR = re.compile(r"v_(readfirstlane|readlane|cmpx?_|add_co|sub_co|addc_co|subb_co|div_scale)")
NO_RESULT = re.compile(r"s_(waitcnt|nop|cbranch|branch|barrier|cmp|bitcmp|setprio|sleep|endpgm|sethalt)")
NO_VECTOR_RESULT = re.compile(r"v_(mfma|cmpx?_|readlane|readfirstlane|nop)")
ACCUMULATION = re.compile(r"v_mfma_(i32_32x32x32_i8|scale_f32_32x32x64_f8f6f4) a\[|v_accvgpr_write_b32 a\d+, 0$|"
                          r"v_accvgpr_read_b32 v\d+, a\d+$")


def code_objects(path):
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


def listings(path):
    """The disassembly of each of them."""
    with tempfile.TemporaryDirectory() as d:
        f = os.path.join(d, "code.o")
        for obj in code_objects(path):
            with open(f, "wb") as out:
                out.write(obj)
            yield subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], stdout=subprocess.PIPE, text=True, check=True).stdout


def kernels(listing):
    """name, instructions and branch targets (by index) of every function in a disassembly."""
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


def _scalars(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"s(\d+)$", operand)
    return {int(m[1])} if m else set()


def _operands(text):
    return [w for part in text.split(None, 1)[1:] for t in part.split(",") for w in t.split()]


def _registers(text, file="v"):
    """Numbers of the vector registers (file "a": accumulation registers) that an instruction names."""
    found = set()
    for lo, hi in re.findall(r"\b%s\[(\d+):(\d+)\]" % file, text):
        found.update(range(int(lo), int(hi) + 1))
    found.update(int(r) for r in re.findall(r"\b%s(\d+)\b" % file, text))
    return found


def _states(text):
    m = re.match(r"s_nop (\d+)", text)
    return int(m[1]) + 1 if m else 1


def _paths_back(code, targets):
    """A function that gives the instructions which may come right before one (targets None: the one above it)."""
    jumps_to = {}
    for at, to in (targets or {}).items():
        jumps_to.setdefault(to, []).append(at)

    def before(k):
        through = k > 0 and (targets is None or not code[k - 1].startswith(("s_branch", "s_endpgm", "s_setpc")))
        return ([k - 1] if through else []) + jumps_to.get(k, [])
    return before


def too_close(code, targets=None):
    """Vector memory instructions that read a scalar register the vector ALU wrote fewer than WAIT_STATES before, on any path."""
    before = _paths_back(code, targets)
    found = []
    for k, text in enumerate(code):
        if not VMEM.match(text):
            continue
        want = set().union(*(_scalars(o) for o in _operands(text)), set())
        todo = [(j, 0, want) for j in before(k) if want]
        while todo:
            j, states, want = todo.pop()
            other = code[j]
            operands = _operands(other)
            if WRITES_SCALAR.match(other):
                # the result is the first operand, or the second of those that have a carry or a condition beside it
                if any(_scalars(o) & want for o in operands[:2] if not other.startswith("v_read") or o is operands[0]):
                    found.append(" ; ".join(code[j:k + 1]) if j < k else "%s ... %s" % (other, text))
                    continue
            elif other.startswith("s_") and not NO_RESULT.match(other) and operands:
                want = want - _scalars(operands[0])   # what is read is the scalar ALU's, which needs no wait
            states += _states(other)
            if want and states < WAIT_STATES:
                todo += [(p, states, want) for p in before(j)]
    return found


def operands_too_close(code, targets):
    """Multiplications that read a register the vector ALU wrote fewer than OPERAND_WAIT_STATES before, on any path."""
    before = _paths_back(code, targets)
    found = []
    for k, text in enumerate(code):
        if not text.startswith("v_mfma"):
            continue
        want = {file: _registers(text, file) for file in "va"}
        todo = [(j, 0) for j in before(k)]
        while todo:
            j, states = todo.pop()
            other = code[j]
            if other.startswith("v_") and not NO_VECTOR_RESULT.match(other):
                result = other if "swap" in other else other.split(",")[0]   # (a swap writes both of its operands)
                if any(_registers(result, file) & want[file] for file in "va"):
                    found.append("%s ... %s" % (other, text))
                    continue
            states += _states(other)
            if states < OPERAND_WAIT_STATES:
                todo += [(p, states) for p in before(j)]
    return found


def in_flight(code, targets):
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


def faults(path):
    """What in the machine code of a library does not hold (see above), as texts."""
    found, tile_gemms = [], 0
    for listing in listings(path):
        for name, code, targets in kernels(listing):
            found += ["%s: scalar register too young: %s" % (name, t) for t in too_close(code, targets)]
            found += ["%s: operand too young: %s" % (name, t) for t in operands_too_close(code, targets)]
            if TILE_GEMM not in name:
                continue
            tile_gemms += sum(t.startswith("v_mfma") for t in code) > 100
            found += ["%s: register under way: %s" % (name, t) for t in in_flight(code, targets)]
            found += ["%s: spilled or called: %s" % (name, t) for t in code if t.startswith(("scratch_", "s_swappc"))]
            found += ["%s: accumulation register: %s" % (name, t) for t in code
                      if re.search(r"\ba(\d+|\[)", t) and not ACCUMULATION.match(t)]
    if tile_gemms != 2:    # int8 and FP8
        found.append("%d kernels of the tile GEMM instead of 2 were looked at" % tile_gemms)
    return found


def check(path):
    """Raises RuntimeError where something does not hold."""
    found = faults(path)
    if found:
        raise RuntimeError("the machine code of %s does not keep what its inline assembly rests on (%d places):\n%s" %
                           (path, len(found), "\n".join(found[:20])))
