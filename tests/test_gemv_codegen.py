"""What the compiler makes of the single-row product's prologue (hipcc cross-compiles here: no GPU needed)."""
import os
import re
import subprocess

from rllama_amd import build

SOURCE = """
#include "gemv_device.h"
using namespace rlh;
__global__ __launch_bounds__(kGemvThreads) void kernel(GemvParams p) {
    extern __shared__ uint4_t smem_raw[];
    __shared__ float red[16];
    gemv_body<half_t, half_t, kEpiSilu, true, kPreSelf>(p, smem_raw, red, nullptr);
}
"""


def test_long_rows_do_not_clear_the_registers_of_the_first_burst(tmp_path):
    """w1|w3 of long rows: the 32 registers of the first burst are written by its loads alone.  Clearing them first costs two moves each (on
    either side of the branch for rows that are shorter than a burst) between the loads of x and those of the burst: 117 registers
    cleared in all, against 52 for the sums, the padding of x and the candidates."""
    src, out = tmp_path / "long_rows.hip", tmp_path / "long_rows.s"
    src.write_text(SOURCE)
    flags = [f for f in build.FLAGS if f != "-fPIC"]
    subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-S", "-I", build.CSRC, str(src), "-o", str(out)], check=True, capture_output=True)
    text = out.read_text()
    cleared = len(re.findall(r"\tv_mov_b32_e32 v\d+, 0\s", text)) + 2 * len(re.findall(r"\tv_mov_b64_e32 v\[\d+:\d+\], (?:0|[vs]\[)", text))
    assert os.path.getsize(out) and "global_load_dwordx4" in text
    assert cleared < 52 + 32
