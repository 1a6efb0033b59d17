"""The addresses of the 3 x 3 convolution kernel that keeps its input rows in LDS (csrc/qconv_walk.hpp), compiled for the host:
every load of every thread lies in the input or is taken for padding, what it puts into LDS lies before the channel parameters,
and every fragment read finds the pixel that its window position has."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "intel-extension-for-tensorflow_amd", "csrc")

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>
namespace itexhip {
@FAST_DIV@
}
#include "qconv_walk.hpp"
using namespace itexhip;

long workgroups = 0, bad = 0;
void fail(const char* what, int c, int b, int h, int w, int oh, int ow, int n, long at) {
  if (++bad < 10) std::printf("%s: C %d B %d in %d x %d out %d x %d N %d at %ld\n", what, c, b, h, w, oh, ow, n, at);
}

template <int PIECES>
void check(int B, int H, int W, int oh, int ow, int pt, int pl, int N) {
  const int C = PIECES * 16, pitch = direct_pitch(C), M = B * oh * ow;
  if ((ow + 2LL) * pitch * 3 > kLdsPerCu) return;
  const DirectPlan plan = plan_direct(M, C, N, oh, ow);
  if (plan.per_wg == 0) return;
  DirectGeometry<FastDiv> s{};
  s.M = M; s.in_h = H; s.in_w = W; s.out_h = oh; s.out_w = ow; s.pad_top = pt; s.pad_left = pl;
  s.by_out_w = make_fast_div(ow); s.by_out_h = make_fast_div(oh);
  set_walk(s, PIECES, make_fast_div);
  s.tiles = (M + 31) / 32;
  s.per_wg = plan.per_wg;
  const long bytes = 1L * B * H * W * C;
  auto pixel = [&](int b, int h, int w) -> long {  // byte of the pixel, -1: padding
    return h < 0 || h >= H || w < 0 || w >= W ? -1 : ((1L * b * H + h) * W + w) * C;
  };
  auto wrong = [&](const char* what, long at) { fail(what, C, B, H, W, oh, ow, N, at); };
  if (1L * plan.wgs * plan.per_wg < s.tiles || 1L * (plan.wgs - 1) * plan.per_wg >= s.tiles) wrong("workgroups", plan.wgs);
  if (plan.panel < 0 || plan.panel % 16 != 0 || plan.lds > kLdsPerCu) wrong("LDS", plan.lds);
  std::vector<long> lds(plan.panel / 16);
  const int stride = plan.wgs <= 6 ? 1 : plan.wgs / 5;
  for (int wg = 0; wg < plan.wgs; wg = wg + stride < plan.wgs || wg == plan.wgs - 1 ? wg + stride : plan.wgs - 1) {
    ++workgroups;
    const int t0 = wg * s.per_wg, t1 = std::min(t0 + s.per_wg, s.tiles), v0 = s.first_row(t0), v1 = s.last_row(t1);
    const int row_pieces = s.wp * PIECES, pieces = (v1 - v0) * row_pieces;
    lds.assign(lds.size(), -2);
    for (int t = 0; t < kDirectThreads; ++t) {
      InputWalk<PIECES, FastDiv> walk(s, v0, t);
      for (int i0 = 0; i0 == 0 || i0 < pieces; i0 += 8 * kDirectThreads)
        for (int u = 0; u < 8; ++u, walk.advance(s)) {
          const int i = i0 + t + u * kDirectThreads;
          long at = -1;
          uint32_t offset;
          if (walk.inside(s, &offset) && i < pieces) at = offset;
          if (at + 16 > bytes) wrong("read", at);
          if (i >= pieces) continue;
          const int v = v0 + i / row_pieces, p = i % row_pieces;
          const long px = pixel(v / s.vr, v % s.vr - pt, p / PIECES - pl);
          if (at != (px < 0 ? -1 : px + p % PIECES * 16)) wrong("piece", i);
          const int slot = piece_at<PIECES>(i) / 16;
          if (slot >= static_cast<int>(lds.size())) wrong("store", slot);
          else lds[slot] = at;
        }
    }
    for (int tile = t0; tile < t1; ++tile)
      for (int l = 0; l < 32; ++l) {
        const int m = std::min(tile * 32 + l, M - 1), at = s.window_at(m, v0, s.wp * pitch, pitch);
        for (int k = 0; k < 9; ++k)
          for (int c = 0; c < PIECES; ++c) {
            const int slot = at / 16 + (k / 3 * s.wp * pitch + k % 3 * pitch) / 16 + c;
            const long px = pixel(m / ow / oh, m / ow % oh - pt + k / 3, m % ow - pl + k % 3);
            if (slot < 0 || slot >= static_cast<int>(lds.size())) wrong("fragment", slot);
            else if (lds[slot] != (px < 0 ? -1 : px + c * 16)) wrong("fragment's pixel", m);
          }
      }
  }
}

int main() {
  std::mt19937 g(1);
  auto below = [&](int n) { return static_cast<int>(g() % n); };
  auto size = [&](int most) { const int r = 1 << below(9); return 1 + below(std::min(r, most)); };
  for (int i = 0; i < 6000; ++i) {
    const int H = size(256), W = size(256), pt = below(3), pl = below(3);
    const int oh = std::max(1, H + pt - 2 + below(4)), ow = std::max(1, W + pl - 2 + below(4));
    int B = 1 + below(40);
    while (B > 1 && 1L * B * oh * ow > 60000) B /= 2;
    const int N = 32 * (1 + below(12));
    switch (i % 4) {
      case 0: check<2>(B, H, W, oh, ow, pt, pl, N); break;
      case 1: check<4>(B, H, W, oh, ow, pt, pl, N); break;
      case 2: check<6>(B, H, W, oh, ow, pt, pl, N); break;
      default: check<8>(B, H, W, oh, ow, pt, pl, N);
    }
  }
  std::printf("%ld workgroups, %ld wrong\n", workgroups, bad);
  return bad != 0 || workgroups < 10000;
}
"""


def fast_div_source():
    src = open(os.path.join(CSRC, "qgemm_common.hpp")).read()
    end = src.index("}\n", src.index("__device__ __forceinline__ int fast_div")) + 2
    return src[src.index("struct FastDiv"):end].replace("__device__ __forceinline__", "inline")


def run(tmp_path, program):
    src, exe = tmp_path / "walk.cc", tmp_path / "walk"
    src.write_text(program.replace("@FAST_DIV@", fast_div_source()))
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout


def test_every_address(tmp_path):
    run(tmp_path, PROGRAM)


PLANS = r"""
#include <cstdint>
#include <cstdio>
namespace itexhip {
@FAST_DIV@
}
#include "qconv_walk.hpp"
using namespace itexhip;
// batch, rows, columns, channels, results, where it measured faster: 1 here, 0 elsewhere
const int cases[][6] = {{32, 56, 56, 64, 64, 1}, {32, 28, 28, 128, 128, 1}, {32, 112, 112, 32, 32, 1}, {1, 14, 14, 32, 32, 1},
                        {4, 62, 62, 128, 224, 1}, {17, 12, 131, 128, 96, 1}, {4, 288, 288, 32, 96, 0}, {11, 253, 253, 32, 96, 0},
                        {3, 195, 195, 96, 224, 0}};
int main() {
  int bad = 0;
  for (const auto& c : cases) {
    const int M = c[0] * c[1] * c[2];
    const DirectPlan p = plan_direct(M, c[3], c[4], c[1], c[2]);
    // workgroups of the busiest XCD's CUs: as many as an even spread gives
    const int busiest = ((p.wgs + 7) / 8 * p.groups_n + 31) / 32, even = (p.wgs * p.groups_n + 255) / 256;
    const bool here = p.us < others_us(M, 9 * c[3], c[4], true);
    if (busiest > even || here != (c[5] == 1)) {
      ++bad;
      std::printf("%d x %d x %d x %d -> %d: %d workgroups x %d, here %d\n", c[0], c[1], c[2], c[3], c[4], p.wgs, p.groups_n, here);
    }
  }
  return bad;
}
"""


def test_run_lengths_and_choice(tmp_path):
    """No run length leaves one XCD with a round of workgroups more than the others; the calls that measured faster elsewhere go
    there."""
    run(tmp_path, PLANS)


SHORTCUTS = r"""
#include <cstdint>
#include <cstdio>
#include <random>
namespace itexhip {
@FAST_DIV@
}
#include "qconv_walk.hpp"
using namespace itexhip;
int main() {
  std::mt19937 g(2);
  auto size = [&](int most) { return 1 + static_cast<int>(g() % (1 + g() % most)); };
  int bad = 0, runs = 0;
  for (int i = 0; i < 20000; ++i) {
    const int B = size(64), oh = size(300), ow = size(300), C = 32 * (1 + static_cast<int>(g() % 4)), N = 32 * size(16);
    if ((ow + 2LL) * direct_pitch(C) * 3 > kLdsPerCu) continue;
    const int64_t M = 1LL * B * oh * ow, tiles = (M + 31) / 32, c32 = C / 32, blocks = N / 32;
    const int64_t waves_n = blocks % 4 == 0 ? 4 : blocks % 2 == 0 ? 2 : 1, groups = blocks / waves_n, waves_m = 4 / waves_n;
    const int64_t resident = c32 == 1 ? 4 : c32 == 2 ? 3 : 2;
    double best = 1e30;
    int64_t per_wg = 0;
    for (int64_t per = 1; per <= kDirectMaxTiles; ++per) {
      const int64_t rows = (32 * per + ow - 2) / ow + 1, images = (rows + oh - 2) / oh;
      const int64_t bytes = (rows + 2 + 2 * images) * (ow + 2) * direct_pitch(C) + 384 * waves_n;
      if (bytes > kLdsPerCu) break;
      const int64_t n = (((tiles + per - 1) / per + 7) / 8 * groups + 31) / 32, at_once = std::min(resident, kLdsPerCu / bytes);
      const double us = static_cast<double>(n) * static_cast<double>((per + waves_m - 1) / waves_m) * (0.18 + 0.2 * static_cast<double>(c32)) *
                            (n == 1 || at_once == 1 ? 1.28 : 1.0) + 3.7 * static_cast<double>((n + at_once - 1) / at_once);
      if (us < best) { best = us; per_wg = per; }
    }
    const DirectPlan p = plan_direct(static_cast<int>(M), C, N, oh, ow);
    runs += per_wg > 1;
    if (p.per_wg != per_wg || (per_wg > 0 && p.wgs != (tiles + per_wg - 1) / per_wg) || p.us < 0) {
      if (++bad < 5) std::printf("%d x %d x %d x %d -> %d: %d, %ld\n", B, oh, ow, C, N, p.per_wg, static_cast<long>(per_wg));
    }
  }
  return bad != 0 || runs < 1000;
}
"""


def test_shortcuts_of_the_run_length(tmp_path):
    """The search that a call pays for finds what the whole one does."""
    run(tmp_path, SHORTCUTS)
