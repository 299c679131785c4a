"""The passes, row tiles and pieces of the fp32 products (rllama_amd/csrc/split3_plan.h), on the CPU over sizes and amounts of work
memory: a product whose first pass has a plan has one for every pass, and nothing outgrows the work memory."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rllama_amd", "csrc")

PROGRAM = r"""
#include "split3_plan.h"
#include <cstdio>
#include <initializer_list>
using namespace rlh;

static int check(int m, int n, int k, int ldc, size_t ws) { // 0: refused at the first pass, 1: fine, -1: a fault
    int passes = 0;
    for (int left = m; left > 0;) {
        const Split3Plan q = plan_split3(left, n, k, ldc, ws, 256);
        if (q.rows == 0 && passes == 0) return 0;
        const size_t partial = q.pieces > 1 ? (size_t)q.pieces * q.rows * n * 4 : 0;
        const int height = q.tiles * 32;
        if (q.rows < 1 || q.rows > left || q.tiles < 1 || q.tiles > 8 || q.m_pad < q.rows || q.m_pad % height != 0 || q.m_pad - q.rows >= 32 * (q.m_pad / height) ||
            q.planes_bytes != (size_t)q.m_pad * k * 6 || q.planes_bytes + partial > ws || q.pieces < 1 || (q.pieces > 1 && k / 32 / q.pieces < 4)) {
            printf("m %d n %d k %d work memory %zu: pass %d of the last %d rows: rows %d tiles %d m_pad %d pieces %d\n", m, n, k, ws, passes, left, q.rows, q.tiles,
                   q.m_pad, q.pieces);
            return -1;
        }
        left -= q.rows;
        passes++;
    }
    return 1;
}

int main() {
    const int ks[] = {32, 96, 4096, 5120, 11008, 13824, 22016, 28672, 32768, 40960, 131072, 131104};
    long fine = 0, refused = 0;
    for (size_t mb : {192, 64})
        for (int k : ks)
            for (int n : {96, 4096, 4098})
                for (int m = 1; m <= 9216; m++) {
                    const int r = check(m, n, k, n, mb << 20);
                    if (r < 0) return 1;
                    // refused only where not even one tile of 256 rows fits
                    if (r == 0 && (mb << 20) >= (size_t)256 * k * 6) return printf("m %d k %d refused\n", m, k), 1;
                    (r ? fine : refused)++;
                }
    // with what split3_work_bytes asks for, for any number of rows up to the one asked for, the plan is that of more work memory
    const size_t most = (size_t)192 << 20;
    for (int k : ks)
        for (int n : {96, 4096, 12288})
            for (int cap : {1, 8, 131, 256, 257, 300, 1345, 2048}) {
                size_t ws = split3_work_bytes(cap, n, k);
                if (ws > most) continue;
                for (int m = 1; m <= cap; m++) {
                    const Split3Plan a = plan_split3(m, n, k, n, ws, 256), b = plan_split3(m, n, k, n, most, 256);
                    if (a.rows != b.rows || a.tiles != b.tiles || a.m_pad != b.m_pad || a.pieces != b.pieces) return printf("m %d of %d n %d k %d: work memory %zu\n", m, cap, n, k, ws), 1;
                }
            }
    printf("%ld fine, %ld refused\n", fine, refused);
    return fine > 0 && refused > 0 ? 0 : 1;
}
"""


def test_every_pass_of_a_product_has_a_plan(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
