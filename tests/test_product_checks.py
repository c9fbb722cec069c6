"""What a product asks of its buffers, on the host: a kernel cannot know how
long they are."""
import os
import re
import shutil
import subprocess
import sys

import pytest
import torch

from ollamamq_amd.ops import hip


@pytest.mark.parametrize("M", [1, 32, 33, 128])
def test_sums_of_whole_row_tiles(M):
    """A product writes sums of squares of 32 rows, so fewer are refused."""
    N, K, rows = 64, 64, -(-M // 32) * 32
    x, w, y = (torch.empty(n, dtype=torch.bfloat16)
               for n in (rows * K, N * K, rows * N))
    with pytest.raises(AssertionError):
        hip.linear_packed(x, w, None, N, K=K, xlds=2, M_frag=M, yfrag=1, y=y,
                          sq_out=torch.empty(rows - 1, N // 32))


SPY = """
#include <stdio.h>
int hipFuncSetAttribute(const void* kernel, int attribute, int value) {
    printf("%p %d\\n", kernel, value);
    return 1;                           /* and so nothing is launched */
}
"""
CALLS = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)     # ahead of HIP's own
from ollamamq_amd.ops import hip
hip.require()
some = 1 << 20                                         # nothing reads it
for hm, hn in (*hip.TILES, hip.TILE_LEAST):
    for epi in (hip.TILE_GATED, hip.TILE_ROPE):
        for M in (129, 9000):
            for nt in (1, 16, 22, 53, 200, 300):
                assert hip._lib.tile_gemm_bf16(
                    some, some, some, some, None, some, some, some, nt, 0.0,
                    0.0, M, 384, 256, epi, hm, hn, 1, 8, 16, 0, 256,
                    *[some] * 7, 1, 1, 16, 1, None)
"""


def test_a_kernel_has_one_limit_of_lds(tmp_path):
    """The limit is the kernel's, not the call's: one that went with the call
    would be another thread's too."""
    if not hip.available():
        pytest.skip("the extension is not built")
    if torch.cuda.is_available():       # a call that got past the spy would run
        pytest.skip("only where there is no device")
    source, spy = tmp_path / "spy.c", tmp_path / "spy.so"
    source.write_text(SPY)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", spy, source], check=True)
    out = subprocess.run([sys.executable, "-c", CALLS, spy], check=True,
                         env={**os.environ, "HIP_VISIBLE_DEVICES": "-1"},
                         capture_output=True, text=True).stdout
    limits = {}
    for line in out.splitlines():
        kernel, value = line.split()
        limits.setdefault(kernel, set()).add(int(value))
    assert len(limits) > 15
    assert all(len(v) == 1 and max(v) <= 160 * 1024 for v in limits.values())


LLVM = "/opt/rocm/llvm/bin"


@pytest.mark.skipif(not os.path.exists(f"{LLVM}/llvm-readelf"),
                    reason="needs ROCm's object tools")
def test_narrow_blocks_keep_their_sums_in_registers(tmp_path):
    """Three blocks a CU leave a lane of k_narrow 80 registers; what does not fit
    would go through memory in the loop that memory bounds."""
    if not hip.available():
        pytest.skip("the extension is not built")
    lib = tmp_path / "kernels.so"
    shutil.copy(hip._lib._name, lib)
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", lib], check=True,
                   capture_output=True)
    found = 0
    for part in tmp_path.glob("*gfx950"):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", part],
                               check=True, capture_output=True, text=True)
        for kernel in notes.stdout.split("- .agpr_count:")[1:]:
            if "k_narrow" in kernel:
                found += 1
                assert re.search(r"\.private_segment_fixed_size: 0\n", kernel)
                assert re.search(r"\.vgpr_spill_count: 0\n", kernel), kernel
    assert found >= 5
