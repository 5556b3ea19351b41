"""No built kernel runs a vector instruction between a conditional's end and the restore of the execution mask there.

A conditional's joining block may be reached with some lanes (or all of them) off, until the execution mask is restored.  The
compiler can drop that restore in favour of an enclosing conditional's, and its register allocator, which runs later, can
then place the reload of a spilled value (from an accumulation register or from scratch memory) or a copy of a register ahead
of the enclosing one: it misses lanes and they go on with whatever the register held.  A store address did, in the
256 x 256 tiles' epilogue for layers without row sums.  Read from the code in the built library, on the CPU.

What the reading cannot see is a joining block that no branch leads to, which the compiler makes of short conditionals: there
the build's switch that keeps every restore is the only guard, so it is checked as well."""
import importlib
import os
import re
import struct
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "cl-eden-kernel_amd", "libedenhip.so")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

# before a block's first change of the mask, whatever that is; and before its restore any vector or memory instruction at all
# (v_readlane moves between scalar registers and a lane, which the mask has no part in: scalar spills)
RELOAD = re.compile(r"v_accvgpr_(read|write|mov)_b32|scratch_load_")
VECTOR = re.compile(r"(v_(?!readlane|writelane)|ds_|global_|buffer_|flat_|scratch_)")


def code_objects(fatbin):
    """the gfx950 code objects of a library's section of offload bundles"""
    at = fatbin.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", fatbin, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", fatbin, entry)
            if b"gfx950" in fatbin[entry + 24:entry + 24 + name] and size:
                yield fatbin[at + offset:at + offset + size]
            entry += 24 + name
        at = fatbin.find(MAGIC, entry)


def listing(code, path):
    with open(path, "wb") as f:
        f.write(code)
    return subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--mcpu=gfx950", path], capture_output=True, text=True, check=True).stdout


def reloads_ahead_of_the_mask(text):
    """(kernel, instruction) for each reload in a joining block ahead of the block's first change of the mask, and for each vector
    instruction ahead of the mask's restore"""
    found, kernel, start, rows = [], None, 0, []

    def finish():
        targets = set()
        for address, op in rows:
            m = re.match(r"s_cbranch_execz (\d+)", op)
            if m:
                offset = int(m[1])
                targets.add(address + 4 + 4 * (offset - 65536 if offset >= 32768 else offset))
        watching, ahead = False, []
        for address, op in rows:
            if address in targets:
                watching, ahead = True, []
            if not watching:
                continue
            if re.match(r"s_c?branch|s_endpgm|s_setpc", op) or re.search(r"\bexec\b|saveexec", op):
                if op.startswith("s_or_b64 exec exec"):
                    found.extend((kernel, a) for a in ahead)
                watching = False
            elif RELOAD.match(op):
                found.append((kernel, op))
                watching = False
            elif VECTOR.match(op):
                ahead.append(op)

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


def test_the_reader_finds_a_misplaced_copy():
    text = """
0000000000001000 <k>:
\ts_and_saveexec_b64 s[0:1], vcc                             // 000000001000: BE802068
\ts_cbranch_execz 1                                          // 000000001004: BF880001
\tv_add_u32_e32 v0, v1, v2                                   // 000000001008: 68000501
\tv_mov_b32_e32 v7, v3                                       // 00000000100C: 7E0E0303
\ts_or_b64 exec, exec, s[2:3]                                // 000000001010: 87FE027E
"""
    assert reloads_ahead_of_the_mask(text) == [("k", "v_mov_b32_e32 v7 v3")]
    # a block that changes the mask otherwise is no joining block's restore: the copy is the next conditional's operand
    assert reloads_ahead_of_the_mask(text.replace("s_or_b64 exec, exec, s[2:3]", "s_and_saveexec_b64 s[2:3], vcc")) == []


def test_no_kernel_runs_ahead_of_the_mask(tmp_path):
    if not os.path.exists(LIBRARY):
        pytest.skip("the library is not built here")
    section = str(tmp_path / "fatbin")
    subprocess.check_call([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + section, LIBRARY, os.devnull])
    with open(section, "rb") as f:
        objects = list(code_objects(f.read()))
    with ThreadPoolExecutor(max_workers=8) as ex:
        texts = list(ex.map(lambda o: listing(o[1], str(tmp_path / str(o[0]))), enumerate(objects)))
    assert sum("s_endpgm" in t for t in texts) >= 10
    assert sum(t.count(">:\n") for t in texts) >= 1000   # kernels
    found = [f for t in texts for f in reloads_ahead_of_the_mask(t)]
    assert not found, found[:10]


def test_every_file_is_built_with_the_restores():
    assert "-amdgpu-remove-redundant-endcf=0" in importlib.import_module("cl-eden-kernel_amd.build").HIP_FLAGS
