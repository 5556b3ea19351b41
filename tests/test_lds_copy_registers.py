"""The direct-to-LDS copies (csrc/eh_internal.h) set m0 inside an asm statement.  The compiler drops a setting of m0 to the
value that it believes is there already, so the statement has to say that it writes the register: otherwise a copy that the
compiler sets up itself would land wherever the last asm statement pointed.  Compiled here, without a GPU."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "cl-eden-kernel_amd")
SOURCE = """
#include "eh_internal.h"
typedef __attribute__((address_space(1))) const uint32_t global_word;
typedef __attribute__((address_space(3))) uint32_t lds_word;
__global__ void copies(const uint32_t *g, uint32_t elsewhere, uint32_t *out) {
    __shared__ uint32_t s[4096];
    __builtin_amdgcn_global_load_lds((global_word *)(g + threadIdx.x), (lds_word *)s, 4, 0, 0);
    %s
    __builtin_amdgcn_global_load_lds((global_word *)(g + 64 + threadIdx.x), (lds_word *)s, 4, 0, 0);
    __syncthreads();
    out[threadIdx.x] = s[threadIdx.x];
}
"""


@pytest.mark.parametrize("copy", ["eh::dma16_off(g, threadIdx.x * 16, elsewhere);", "eh::dma16(g + threadIdx.x * 4, elsewhere);"])
def test_the_compilers_own_copies_set_m0_again(tmp_path, copy):
    source, listing = tmp_path / "copies.hip", tmp_path / "copies.s"
    source.write_text(SOURCE % copy)
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-O3", "-std=c++17", "-w", "-I" + os.path.join(ROOT, "include"),
                           "-I" + os.path.join(PKG, "csrc"), "-S", "--cuda-device-only", str(source), "-o", str(listing)])
    steps = re.findall(r"s_mov_b32 (m0), (\S+)|(global_load_lds_\w+)", listing.read_text())
    held, at = None, []
    for register, value, load in steps:
        if register:
            held = value
        else:
            at.append((load, held))
    assert [load for load, _ in at] == ["global_load_lds_dword", "global_load_lds_dwordx4", "global_load_lds_dword"]
    assert at[0][1] == at[2][1] != at[1][1], at
