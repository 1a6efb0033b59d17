"""The offsets of the BatchMatMul kernel's unaligned loads (csrc/qbmm_reads.hpp), compiled for the host: for every thread of a
workgroup and every tile, the first loads included that precede the K loop, the bytes lie inside the operand."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "qbmm_reads.hpp"
using namespace itexhip;
int main() {
  const int64_t sizes[] = {0, 1, 2, 3, 4, 5, 7, 15, 16, 17, 31, 63, 64, 65, 79, 130, 197};
  long fits = 0, bad = 0;
  for (int64_t R : sizes) for (int64_t K : sizes) for (int k_fastest = 0; k_fastest < 2; ++k_fastest) {
    if (R == 0 || !vector_reads_fit(k_fastest, R, K)) continue;
    ++fits;
    for (int64_t r0 = 0; r0 < (R + 127) / 128 * 128; r0 += 64)
      for (int64_t k0 = 0; k0 == 0 || k0 < K; k0 += 64)
        for (int t = 0; t < 256; ++t)
          for (int i = 0; i < (k_fastest ? 1 : 4); ++i) {
            const int64_t at = k_fastest ? read_offset_k_fastest(r0 + (t >> 2), k0 + (t & 3) * 16, R, K)
                                         : read_offset_r_fastest(r0 + (t & 15) * 4, k0 + (t >> 4) * 4 + i, R, K);
            if (at < 0 || at + (k_fastest ? 16 : 4) > R * K) {
              if (++bad < 5) std::printf("R %ld K %ld k_fastest %d: offset %ld\n", (long)R, (long)K, k_fastest, (long)at);
            }
          }
  }
  std::printf("%ld shapes, %ld reads outside\n", fits, bad);
  return bad != 0 || fits < 100;
}
"""


def test_every_read_lies_inside_the_operand(tmp_path):
    src, exe = tmp_path / "reads.cc", tmp_path / "reads"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "intel-extension-for-tensorflow_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout
