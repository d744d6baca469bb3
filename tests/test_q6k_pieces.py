"""The 16-byte pieces that the Q6_K tile kernels copy stay inside the matrix:
host-compiled sweep over the kernels' own address arithmetic
(csrc/kernels/q6k_pieces.hpp), matrices at every allowed alignment."""
import os
import subprocess

KERNELS = os.path.join(os.path.dirname(__file__), "..", "citlali-llm-engine_amd", "csrc", "kernels")

SWEEP = r"""
#include <stdio.h>
#include "q6k_pieces.hpp"
using namespace citlali::hip;
int main() {
    long long outside = 0, at_ends = 0, pieces = 0;
    for (uintptr_t w = 4096; w < 4112; w += 4)                  // Q6_K weights are 4-byte aligned
        for (int nb = 1; nb <= 112; nb = nb < 20 ? nb + 1 : nb + 23)
            for (int rows = 1; rows <= 50; ++rows) {
                const int row_bytes = nb * kQ6KBlockBytes;
                const uintptr_t end = w + (uintptr_t)rows * row_bytes;
                for (int first = 0; first < rows; first += 16) {
                    const int n = rows - first < 16 ? rows - first : 16;
                    const Q6KEnds e = q6k_ends(w, rows, nb, first == 0, first + n == rows);
                    for (int b = 0; b < nb; ++b) {
                        const uintptr_t base = w + (uintptr_t)first * row_bytes + (uintptr_t)b * kQ6KBlockBytes;
                        const int skew = (int)(base & 15);
                        for (int r = 0; r < n; ++r) {
                            const uintptr_t block = base + (uintptr_t)r * row_bytes;
                            for (int p = 0; p < kQ6KPieces; ++p, ++pieces) {
                                const uintptr_t at = base - skew + q6k_piece(skew, r * row_bytes, p);
                                if (at % 16) return printf("misaligned\n"), 1;
                                if (at + 16 <= block || at >= block + kQ6KBlockBytes) return printf("idle piece\n"), 1;
                                if (p == 0 && at > block) return printf("block begins before its pieces\n"), 1;
                                if (p + 1 == kQ6KPieces && at + 16 < block + kQ6KBlockBytes) return printf("block ends behind its pieces\n"), 1;
                                if (at >= w && at + 16 <= end) continue;
                                if (b == e.lo || b == e.hi) ++at_ends;   // these go through registers, inside the matrix
                                else ++outside;
                            }
                        }
                    }
                }
            }
    printf("%lld pieces, %lld outside, %lld at the ends\n", pieces, outside, at_ends);
    return outside != 0 || at_ends == 0;
}
"""


def test_pieces_stay_inside_the_matrix(tmp_path):
    src, exe = tmp_path / "pieces.cpp", tmp_path / "pieces"
    src.write_text(SWEEP)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", KERNELS, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
