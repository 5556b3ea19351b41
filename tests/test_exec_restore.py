"""No built kernel reloads a spilled register where lanes that need it are switched off.

A conditional's joining block may be reached with some lanes (or all of them) off, until the execution mask is restored.  The
compiler can drop that restore in favour of an enclosing conditional's, and its register allocator, which runs later, can
then place the reload of a spilled value (from an accumulation register or from scratch memory) ahead
of the enclosing one: the reload misses lanes and they go on with whatever the register held.  A store address did, in the
256 x 256 tiles' epilogue for layers without row sums.  Read from the built code, on the CPU."""
import glob
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJECTS = os.path.join(ROOT, "cl-eden-kernel_amd", "build")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")

RELOAD = re.compile(r"v_accvgpr_(read|write|mov)_b32|scratch_load_")   # (plain moves also merge values at joins, which is sound)


def listing(obj, where):
    """the disassembly of the object's gfx950 code, or "" for an object without kernels"""
    base = os.path.join(where, os.path.basename(obj))
    if subprocess.run([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + base + ".fb", obj, os.devnull], capture_output=True).returncode:
        return ""
    subprocess.check_call([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", "--input=" + base + ".fb",
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--output=" + base + ".co"])
    return subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--mcpu=gfx950", base + ".co"], capture_output=True, text=True, check=True).stdout


def reloads_ahead_of_the_mask(text):
    """(kernel, instruction) for each reload in a joining block that stands ahead of the block's first change of the mask"""
    found, kernel, start, rows = [], None, 0, []

    def finish():
        targets = set()
        for address, op in rows:
            m = re.match(r"s_cbranch_execz (\d+)", op)
            if m:
                offset = int(m[1])
                targets.add(address + 4 + 4 * (offset - 65536 if offset >= 32768 else offset))
        watching = False
        for address, op in rows:
            if address in targets:
                watching = True
            if not watching:
                continue
            if re.match(r"s_c?branch|s_endpgm|s_setpc", op) or re.search(r"\bexec\b|saveexec", op):
                watching = False
            elif RELOAD.match(op):
                found.append((kernel, op))
                watching = False

    for line in text.splitlines():
        m = re.match(r"([0-9a-f]+) <(\S+)>:", line)
        if m:
            finish()
            kernel, rows = m[2], []
            continue
        m = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):", line)
        if m:
            rows.append((int(m[2], 16), re.sub(r"\s+", " ", m[1]).replace(",", "")))
    finish()
    return found


def test_the_reader_finds_a_misplaced_reload():
    text = """
0000000000001000 <k>:
\ts_and_saveexec_b64 s[0:1], vcc                             // 000000001000: BE802068
\ts_cbranch_execz 1                                          // 000000001004: BF880001
\tv_add_u32_e32 v0, v1, v2                                   // 000000001008: 68000501
\tv_accvgpr_read_b32 v119, a3                                // 00000000100C: D3D84077
\ts_or_b64 exec, exec, s[2:3]                                // 000000001014: 87FE027E
"""
    assert reloads_ahead_of_the_mask(text) == [("k", "v_accvgpr_read_b32 v119 a3")]
    assert reloads_ahead_of_the_mask(text.replace("100C", "1012").replace("1014", "100C")) == []   # behind the restore


def test_no_kernel_reloads_ahead_of_the_mask(tmp_path):
    objects = sorted(glob.glob(os.path.join(OBJECTS, "*.o")))
    if not objects:
        pytest.skip("the objects of a build are not here")
    with ThreadPoolExecutor(max_workers=8) as ex:
        texts = list(ex.map(lambda o: listing(o, str(tmp_path)), objects))
    assert sum("s_endpgm" in t for t in texts) >= 10
    found = [f for t in texts for f in reloads_ahead_of_the_mask(t)]
    assert not found, found[:10]
