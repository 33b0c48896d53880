"""The built kernels keep a wait that the hardware does not: a vector-memory instruction must not read a scalar register
within five wait states of a vector instruction that wrote it (v_readfirstlane, v_readlane of a spilled scalar, a compare).
The compiler keeps that distance for instructions of its own, not for those written in inline assembly, whose scalar base
may come out of such an instruction right in front of the statement.  A base read too early is a wild address, now and
then; so the machine code of the library that was built here is looked through, along branches too."""
import os
import re
import shutil
import subprocess

import pytest

from flaggems_amd import _lib

WAIT_STATES = 5
_LINE = re.compile(r"^\t(\S+)(?: (.*?))?\s*// ([0-9A-F]+):")
_TARGET = re.compile(r"<(\S+?)(?:\+0x([0-9a-f]+))?>\s*$")
_MEMORY = re.compile(r"(global|buffer|flat|scratch)_")


def _scalars(operand):
    """Numbers of the scalar registers that an operand names (vcc: 106, 107)."""
    operand = operand.strip()
    if operand in ("vcc", "vcc_lo", "vcc_hi"):
        return {"vcc": {106, 107}, "vcc_lo": {106}, "vcc_hi": {107}}[operand]
    m = re.match(r"s\[(\d+):(\d+)\]$|s(\d+)$", operand.split(" ")[0])
    if not m:
        return set()
    return {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))


def _parse(listing):
    """[(mnemonic, operands, address)] and, for branches, the target's address beside the index."""
    code, jumps, symbols = [], [], {}
    for line in listing.splitlines():
        m = re.match(r"^([0-9a-f]{16}) <(\S+)>:", line)
        if m:
            symbols[m[2]] = int(m[1], 16)
            continue
        m = _LINE.match(line)
        if not m:
            continue
        name, rest = m[1], m[2] or ""
        if name.startswith(("s_branch", "s_cbranch")):
            t = _TARGET.search(line)
            if t:
                jumps.append((len(code), t[1], int(t[2] or "0", 16)))
        code.append((name, [] if not rest else re.split(r",\s*", rest), int(m[3], 16)))
    return code, [(i, symbols[s] + o) for i, s, o in jumps if s in symbols]


def _states(name, operands):
    return int(operands[0], 0) + 1 if name == "s_nop" else 1


def _written(name, operands):
    """Scalar registers that a vector instruction writes."""
    if not name.startswith("v_") or not operands:
        return set()
    out = _scalars(operands[0])
    if len(operands) > 1 and ("_co_" in name or "div_scale" in name or "mad_u64" in name or "mad_i64" in name):
        out |= _scalars(operands[1])
    return out


def _faults(listing):
    code, jumps = _parse(listing)
    found = []

    def window(i):  # writes that are still too close in front of instruction i, in layout order
        out, passed = [], 0
        while i > 0 and passed < WAIT_STATES:
            i -= 1
            if code[i][0] in ("s_branch", "s_endpgm", "s_setpc_b64"):
                break
            w = _written(*code[i][:2])
            if w:
                out.append((w, passed, i))
            passed += _states(*code[i][:2])
        return out

    def check(i, recent):  # recent: (registers, wait states passed before instruction i, index of the write)
        name, operands, address = code[i]
        if not _MEMORY.match(name):
            return
        used = set().union(set(), *[_scalars(o) for o in operands])
        for w, passed, at in recent:
            if w & used and passed < WAIT_STATES:
                found.append("%x: %s %s after %s" % (address, name, ", ".join(operands), code[at][0]))

    for i, (name, _, _) in enumerate(code):
        if _MEMORY.match(name):
            check(i, window(i))
    index = {a: i for i, (_, _, a) in enumerate(code)}
    for at, target in jumps:
        recent = [(w, passed + 1, k) for w, passed, k in window(at)]  # (+ 1: the branch)
        i, more = index.get(target), 0
        while recent and i is not None and i < len(code) and more < WAIT_STATES:
            check(i, [(w, passed + more, k) for w, passed, k in recent])
            more += _states(*code[i][:2])
            i += 1
    return found


def _objdump():
    for exe in (shutil.which("llvm-objdump"), "/opt/rocm/llvm/bin/llvm-objdump", "/opt/rocm/lib/llvm/bin/llvm-objdump"):
        if exe and os.path.exists(exe):
            return exe
    pytest.skip("llvm-objdump (part of the toolchain that builds the library) not found")


def _listings(library, folder):
    exe = _objdump()
    copy = os.path.join(str(folder), "lib.so")
    shutil.copy(library, copy)
    subprocess.run([exe, "--offloading", copy], check=True, stdout=subprocess.DEVNULL, cwd=str(folder))
    objects = sorted(f for f in os.listdir(str(folder)) if f.endswith("gfx950"))
    for name in objects:
        yield name, subprocess.run([exe, "-d", "--no-show-raw-insn", os.path.join(str(folder), name)], check=True, text=True,
                                   stdout=subprocess.PIPE).stdout


def test_built_kernels_keep_the_distance(tmp_path):
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("shared library not built on this host")
    seen = 0
    for name, listing in _listings(_lib.LIB_PATH, tmp_path):
        seen += len(_MEMORY.findall(listing))
        assert _faults(listing) == [], name
    assert seen > 10000  # (the listing was understood)


def test_the_check_itself():
    def lines(*ins):
        return "\n".join(["0000000000001000 <k>:"] + ["\t%s// %012X: " % (s.ljust(60), 0x1000 + 4 * i) for i, s in enumerate(ins)])

    load = "global_load_dwordx4 v[0:3], v4, s[6:7] sc1"
    assert len(_faults(lines("v_readfirstlane_b32 s7, v1", "s_nop 0", load))) == 1
    assert len(_faults(lines("v_readlane_b32 s6, v1, 3", "s_nop 3", load))) == 1
    assert not _faults(lines("v_readlane_b32 s6, v1, 3", "s_nop 4", load))
    assert not _faults(lines("v_readlane_b32 s8, v1, 3", load))
    assert len(_faults(lines("v_cmp_lt_i32_e64 s[6:7], v1, v2", "v_mov_b32_e32 v0, 0", load))) == 1
    assert len(_faults(lines("v_cmp_lt_i32_e32 vcc, 0, v2", "global_load_lds_dword v1, vcc"))) == 1
    # over a branch, taken or not
    jump = lines("v_readfirstlane_b32 s7, v1", "s_cbranch_scc1 2", "s_nop 4", load, load).replace("s_cbranch_scc1 2".ljust(60) + "// 000000001004: ",
                 "s_cbranch_scc1 2".ljust(60) + "// 000000001004: BF850002 <k+0x10>")
    assert len(_faults(jump)) == 1
