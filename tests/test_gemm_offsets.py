"""Where the products' operand reads may go (csrc/gemm_offsets.h), by enumeration on the host: a lane's read lies inside its
operand or is refused by the descriptor's range check, also in the steps that are asked for past the contraction's end."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turbot5_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "gemm_offsets.h"
using namespace t5a;
// lines x width elements; the contraction K runs along a line (col 0) or over the lines (col 1)
static long check(int rows, int K, int64_t ld, int size, bool col) {
    const int bytes = operand_bytes(col ? K : rows, col ? rows : K, ld, size), step = step_bytes(K, col ? ld : 1, size);
    if (bytes <= 0 || step < 0) return 1;
    long bad = 0;
    const int steps = (K + kGemmStep - 1) / kGemmStep;
    for (int kk : {0, 1, steps - 2, steps - 1, steps, steps + 1, steps + 4, steps + 8}) {
        if (kk < 0) continue;
        const int64_t scalar = step_offset(kk, K, step);
        bad += scalar < 0 || scalar >= bytes;                       // (the check's difference does not wrap)
        for (int k = 0; k < kGemmStep; k += col ? 1 : 8)
            for (int row : {0, rows / 16 * 8, rows - 8}) {
                if (row < 0) row = 0;
                const int64_t at = (col ? (int64_t)(k < K - 1 ? k : K - 1) * ld + row : row * ld + k) * size;
                const bool wanted = kk < steps && k < K - kk * kGemmStep;
                if (wanted) bad += at > 0x7fffffff;
                const int64_t lane = lane_offset(k, kk, K, (int)at);
                for (int e = 0; e < 8 * size; e += 16) {
                    const bool read = lane + e < bytes - scalar;
                    bad += read != wanted || lane + e > 0x7fffffff || (read && scalar + lane + e + 16 > bytes);
                }
            }
    }
    return bad;
}
int main() {
    long bad = 0, n = 0;
    for (int size : {2, 4})
        for (int rows : {8, 64, 72, 512, 2048, 32128})
            for (int K : {1, 3, 8, 31, 32, 33, 40, 64, 512, 1000, 2048, 4500})
                for (bool col : {false, true}) {
                    if (!col && K % 8) continue;
                    const int64_t width = (col ? rows : K) + 7 & ~7, lines = col ? K : rows, most = (0x7ff00000LL - 1) / (lines * size) / 8 * 8;
                    for (int64_t ld : {width, width + 8, most})      // (the widest lines the entry point takes)
                        if (ld >= width && lines * ld * size < 0x7ff00000LL) { bad += check(rows, K, ld, size, col); ++n; }
                }
    std::printf("%ld %ld\n", n, bad);
    return bad != 0 || n < 300;
}
"""


def test_reads_stay_in_the_operand(tmp_path):
    src, exe = tmp_path / "offsets.cpp", tmp_path / "offsets"
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout + run.stderr
