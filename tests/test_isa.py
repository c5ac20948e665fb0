"""The machine code of the library's kernels: forms that this GPU executes wrongly stay out of it."""
import os
import re
import subprocess

import pytest

from binarybrain_amd.build import LIB_PATH

LLVM = "/opt/rocm/llvm/bin"


def shifts_by_the_last_register(disassembly, allocated):
    """(kernel, instruction) of every 64-bit shift whose amount is in the last vector register that its kernel allocates (in groups of eight).  The GPU reads
    a register pair for the amount, and where the second one does not exist it shifts by v0: wrong results without an error."""
    found, name = [], None
    for line in disassembly:
        m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if m:
            name = m.group(1)
            continue
        m = re.match(r"\s+(v_(?:lshlrev_b64|lshrrev_b64|ashrrev_i64)\S* v\[\d+:\d+\], v(\d+), \S+)", line)
        if m and name in allocated and int(m.group(2)) == (allocated[name] + 7) // 8 * 8 - 1:
            found.append((name, m.group(1)))
    return found


def test_the_check_finds_what_it_looks_for():
    text = ["0000 <k>:", "\tv_lshrrev_b64 v[78:79], v87, s[50:51]   // 1", "\tv_lshrrev_b64 v[78:79], v86, s[50:51]   // 2", "\tv_lshlrev_b64 v[2:3], 2, v[86:87]   // 3"]
    assert len(shifts_by_the_last_register(text, {"k": 88})) == 1 and len(shifts_by_the_last_register(text, {"k": 85})) == 1
    assert not shifts_by_the_last_register(text, {"k": 89})


def lds_loads_behind_a_write_of_m0(disassembly):
    """(kernel, instruction) of every load from memory to LDS that follows a scalar write of M0 at once.  The load takes its LDS address from M0 and must be a wait
    state apart (the compiler sees to that in its own code, not within inline assembly): a stale M0 sends the data elsewhere without an error."""
    found, name, before = [], None, ""
    for line in disassembly:
        m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if m:
            name, before = m.group(1), ""
            continue
        m = re.match(r"\s+(\S+)\s*([^/]*)", line)
        if not m:
            continue
        if re.match(r"(buffer|global)_load", m.group(1)) and (re.search(r"\blds\b", m.group(2)) or "_lds_" in m.group(1)) and re.match(r"s_\S+ m0\b", before):
            found.append((name, line.strip()))
        before = m.group(1) + " " + m.group(2)
    return found


def test_the_check_of_lds_loads_finds_what_it_looks_for():
    load = "\tbuffer_load_dwordx4 v3, s[28:31], s1 offen lds            // 2"
    assert len(lds_loads_behind_a_write_of_m0(["0000 <k>:", "\ts_mov_b32 m0, s21     // 1", load])) == 1
    assert not lds_loads_behind_a_write_of_m0(["0000 <k>:", "\ts_mov_b32 m0, s21     // 1", "\ts_nop 0     // 1", load, "\ts_mov_b32 m0, s2", "0001 <l>:", load])
    assert not lds_loads_behind_a_write_of_m0(["0000 <k>:", "\ts_mov_b32 m0, s21     // 1", "\tbuffer_load_dwordx4 v[0:3], v3, s[28:31], s1 offen   // 2"])


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """the library's code object for the GPU"""
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-objdump", "llvm-readelf")]
    if not os.path.exists(LIB_PATH) or not all(os.path.exists(t) for t in tools):
        pytest.skip("needs the built library and the LLVM tools of ROCm")
    objcopy, bundler = tools[:2]
    at = tmp_path_factory.mktemp("isa")
    fat, out = str(at / "fat"), str(at / "code.o")
    subprocess.run([objcopy, "--dump-section", ".hip_fatbin=" + fat, LIB_PATH, os.devnull], check=True, capture_output=True)
    subprocess.run([bundler, "--unbundle", "--type=o", "--input=" + fat, "--output=" + out, "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True,
                   capture_output=True)
    return out


def disassembly_of(code):
    return subprocess.Popen([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", code], stdout=subprocess.PIPE, text=True)


def test_no_64_bit_shift_by_the_last_register(code):
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", code], check=True, capture_output=True, text=True).stdout
    allocated, name = {}, None
    for line in notes.splitlines():
        m = re.match(r"\s+\.name:\s+(_Z\S+)", line)
        if m:
            name = m.group(1)
        m = re.match(r"\s+\.vgpr_count:\s+(\d+)", line)
        if m:
            allocated[name] = int(m.group(1))
    assert len(allocated) > 300
    text = disassembly_of(code)
    found = shifts_by_the_last_register(text.stdout, allocated)
    assert text.wait() == 0 and not found, found[:5]


def test_lds_loads_are_a_wait_state_behind_their_address(code):
    text = disassembly_of(code)
    found = lds_loads_behind_a_write_of_m0(text.stdout)
    assert text.wait() == 0 and not found, (len(found), found[:5])
