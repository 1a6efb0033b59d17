// Where the 3 x 3 convolution kernel (qconv_direct.hip) puts input rows into LDS and reads them, how many row tiles a workgroup
// takes, and which convolutions are its.  Plain C++: the CPU test of all of it includes this file.  D is the division by a number
// fixed per launch, fast_div(n, D).
#ifndef ITEXHIP_QCONV_WALK_HPP_
#define ITEXHIP_QCONV_WALK_HPP_

#include <stdint.h>

#include <algorithm>

#ifndef ITEXHIP_HD
#ifdef __HIP__
#define ITEXHIP_HD __host__ __device__ inline
#else
#define ITEXHIP_HD inline
#endif
#endif

namespace itexhip {

constexpr int kLdsPerCu = 160 * 1024;
constexpr int kDirectThreads = 256;
constexpr int kDirectMaxTiles = 24;  // of a workgroup

// The output positions stand one after the other, rows of one image after those of the image before it; so do the padded
// images.  A tile is 32 positions.
template <class D>
struct DirectGeometry {
  int M;
  int in_h, in_w, out_h, out_w;
  int pad_top, pad_left;
  int wp, vr;         // input columns, and rows of one image, that windows touch, padding included
  D by_out_w, by_out_h, by_row_pieces, by_vr;
  int step_p, step_h, step_image;  // kDirectThreads pieces of 16 bytes on: pieces of a row, rows of an image, images
  int tiles, per_wg;  // row tiles of 32; of a workgroup

  // row of the padded images in which the windows of output row g begin
  ITEXHIP_HD int window_row(int g) const {
    const int b = fast_div(g, by_out_h);
    return b * vr + (g - b * out_h);
  }
  // rows of the padded images that tiles t0 .. t1 - 1 touch: [first, last)
  ITEXHIP_HD int first_row(int t0) const { return window_row(fast_div(t0 * 32, by_out_w)); }
  ITEXHIP_HD int last_row(int t1) const { return window_row(fast_div((t1 * 32 < M ? t1 * 32 : M) - 1, by_out_w)) + 3; }
  // byte in LDS at which the window of position m begins, v0 being the first row there; bytes of a row and of a pixel
  ITEXHIP_HD int window_at(int m, int v0, int row_bytes, int pitch) const {
    const int g = fast_div(m, by_out_w);
    return (window_row(g) - v0) * row_bytes + (m - g * out_w) * pitch;
  }
};

// the members that follow from out_h and out_w; `pieces` of 16 bytes per pixel
template <class D, class MakeDiv>
void set_walk(DirectGeometry<D>& s, int pieces, MakeDiv make_div) {
  s.wp = s.out_w + 2;
  s.vr = s.out_h + 2;
  const int row_pieces = s.wp * pieces, step = kDirectThreads / row_pieces;
  s.by_row_pieces = make_div(row_pieces);
  s.by_vr = make_div(s.vr);
  s.step_p = kDirectThreads % row_pieces;
  s.step_image = step / s.vr;
  s.step_h = step % s.vr;
}

// A thread's way through the 16-byte pieces of the padded rows from v0 on, kDirectThreads at a time; PIECES per pixel.  The
// divisions are paid once, then counters carry over rows and images.
template <int PIECES, class D>
struct InputWalk {
  int ih, image, p;  // row of an image (pad_top of them above it), image, piece of that row
  ITEXHIP_HD InputWalk(const DirectGeometry<D>& s, int v0, int thread) {
    const int r = fast_div(thread, s.by_row_pieces);
    p = thread - r * (s.wp * PIECES);
    image = fast_div(v0 + r, s.by_vr);
    ih = v0 + r - image * s.vr;
  }
  // Whether the piece lies in the input and not in its padding, and its byte offset then (input bytes < 2^31).  (The caller looks
  // whether there is a piece: behind the last one there may be no image either.)
  ITEXHIP_HD bool inside(const DirectGeometry<D>& s, uint32_t* offset) const {
    const int h = ih - s.pad_top, q = p - s.pad_left * PIECES;
    *offset = static_cast<uint32_t>((image * s.in_h + h) * (s.in_w * PIECES) + q) * 16u;
    return (static_cast<unsigned>(h) < static_cast<unsigned>(s.in_h)) &  // (no branch)
           (static_cast<unsigned>(q) < static_cast<unsigned>(s.in_w * PIECES));
  }
  ITEXHIP_HD void advance(const DirectGeometry<D>& s) {
    p += s.step_p;
    ih += s.step_h;
    image += s.step_image;
    const bool next_row = p >= s.wp * PIECES;
    p -= next_row ? s.wp * PIECES : 0;
    ih += next_row ? 1 : 0;
    const bool next_image = ih >= s.vr;
    ih -= next_image ? s.vr : 0;
    image += next_image ? 1 : 0;
  }
};

// byte of piece i in LDS: pixels lie an odd number of pieces apart, so that the reads of 16 neighbours fall into different banks
template <int PIECES>
ITEXHIP_HD int piece_at(int i) { return (i + i / PIECES) * 16; }
constexpr int direct_pitch(int in_c) { return in_c + 16; }  // of a pixel in LDS

struct DirectPlan {
  int waves_n;   // wavefronts side by side along the channels: 1, 2 or 4
  int groups_n;  // workgroups along them
  int per_wg;    // tiles of a workgroup; 0: rows too wide for LDS
  int wgs;       // workgroups along the positions
  int panel;     // offset in LDS of the channel parameters
  int lds;       // bytes of LDS of a workgroup
  double us;     // estimate of the launch
};

// M > 0, M * N < 2^31, three padded rows fit LDS
inline DirectPlan plan_direct(int M, int in_c, int N, int out_h, int out_w) {
  DirectPlan s{};
  const int blocks = N / 32, c32 = in_c / 32, wp = out_w + 2, pitch = direct_pitch(in_c);
  s.waves_n = blocks % 4 == 0 ? 4 : blocks % 2 == 0 ? 2 : 1;
  s.groups_n = blocks / s.waves_n;
  const int waves_m = 4 / s.waves_n, panel = 12 * 32 * s.waves_n;  // bytes of the channel parameters
  const int tiles = static_cast<int>((static_cast<int64_t>(M) + 31) / 32), resident = c32 == 1 ? 4 : c32 == 2 ? 3 : 2;  // (registers)
  // The tiles of a workgroup: the smallest estimate, us, fitted to 20 shapes (56 x 56 x 64 to 112 x 112 x 32, 1 to 64 images,
  // 64 to 512 results).  A wavefront takes 0.18 + 0.2 per 32 channels for a tile, a CU with one workgroup 1.28 times that, since
  // nothing runs under its waits, and every set of workgroups that a CU holds at once 3.7 for its start.  Workgroups are counted
  // on the busiest XCD: 35 x 7 of them are fewer than 256, but five of the 35 go to one XCD, 35 workgroups to its 32 CUs
  // (4 x 62 x 62 x 128 -> 224: 19.2 us, 12.0 with a shorter run).  Over 2200 shapes of 4 x 4 to 300 x 300 with 13 lengths each the
  // choice is 0.9 % above the best in the mean, 11 % for one in a hundred, 24 % at most.
  double best = 1e30;
  for (int per = 1; per <= kDirectMaxTiles; ++per) {
    // 32 * per positions lie in at most `rows` output rows, which cross `images` borders (two more input rows each)
    const unsigned rows = static_cast<unsigned>(32 * per + out_w - 2) / static_cast<unsigned>(out_w) + 1;
    const unsigned images = rows < 2 ? 0 : rows <= static_cast<unsigned>(out_h) + 1 ? 1 : (rows - 2) / static_cast<unsigned>(out_h) + 1;
    const int64_t staged = static_cast<int64_t>(rows + 2 + 2 * images) * wp;  // pixels put into LDS
    const int64_t bytes = staged * pitch + panel;
    if (bytes > kLdsPerCu) break;
    const unsigned wgs = static_cast<unsigned>(tiles + per - 1) / static_cast<unsigned>(per);
    const int64_t n = (static_cast<int64_t>((wgs + 7) / 8) * s.groups_n + 31) / 32;  // workgroups of the busiest CU
    const int at_once = std::min(resident, static_cast<int>(static_cast<unsigned>(kLdsPerCu) / static_cast<unsigned>(bytes)));
    const int turns = (per + waves_m - 1) / waves_m;  // tiles of a wavefront
    const double sets = n <= at_once ? 1.0 : static_cast<double>((n + at_once - 1) / at_once);
    const double us = static_cast<double>(n) * turns * (0.18 + 0.2 * c32) * (n == 1 || at_once == 1 ? 1.28 : 1.0) + 3.7 * sets;
    if (us < best) {
      best = us;
      s.per_wg = per; s.lds = static_cast<int>(bytes); s.wgs = static_cast<int>(wgs);
      // The launch as a whole, for others_us to be compared with: 2.0, and per set its start, 0.99 for every eight loads per
      // thread that put rows into LDS, and the tiles, 0.86 of whose time adds up for workgroups that share a CU.  Within 10 %
      // (one standard deviation) of 25900 times.
      const double pieces = static_cast<double>(staged * (in_c / 16));
      s.us = 2.0 + sets * (1.06 + 0.99 / (8 * kDirectThreads) * pieces + std::min(turns, (tiles + waves_m - 1) / waves_m) * (0.2 + 0.22 * c32) *
                                      (1.0 + 0.86 * (static_cast<double>(std::min<int64_t>(n, at_once)) - 1.0)));
    }
    if (n == 1) break;  // longer runs leave CUs without one
  }
  s.panel = s.lds - panel;
  return s;
}

// ---- the other kernels for a convolution: [M, K] patches, N results

// Tile shape of the implicit GEMM: the one with the smallest estimated time, rounds of workgroups over the 256 CUs x tile area x
// a penalty for the operand traffic per MFMA of smaller tiles.
inline int pick_conv_tile(int64_t M, int64_t N) {
  struct Shape { int bm, bn; double penalty; };
  static constexpr Shape shapes[3] = {{256, 128, 1.08}, {128, 128, 1.2}, {64, 64, 1.8}};
  int best = 0;
  double best_cost = 1e300;
  for (int i = 0; i < 3; ++i) {
    const int64_t tiles = ((M + shapes[i].bm - 1) / shapes[i].bm) * ((N + shapes[i].bn - 1) / shapes[i].bn);
    const double cost = static_cast<double>((tiles + 255) / 256) * shapes[i].bm * shapes[i].bn * shapes[i].penalty;
    if (cost < best_cost) { best_cost = cost; best = i; }
  }
  return best;
}

// Whether a convolution goes to the kernel for a short K (qgemm_stream.hip, where the reasons stand): quarter_rounds is how often
// its 32 x 64 pieces fill a quarter of the device.
inline bool conv_streams(int64_t K, int64_t N, bool sum, int64_t quarter_rounds) {
  auto within = [&](int64_t least, int64_t most = INT64_MAX) { return quarter_rounds >= least && quarter_rounds <= most; };
  const bool wide = N > 64;
  const int64_t least = sum || K <= 160 || !wide ? 3 : K > 256 && K < 384 && N > 256 && N <= 384 ? 24 : N > 256 || K >= 384 ? 6 : 3;
  return K <= (wide ? 384 : 448) ? within(least) : K <= 448 && (sum ? within(3, 7) : within(6, 7));
}

// Time of a 3 x 3 convolution over 32 to 128 channels on the kernel that would take it, us: fitted to 2200 shapes (tile shapes, one
// standard deviation 4 to 7 %) and 550 (the kernel for a short K, 10 %: 32 x 64 results per wavefront and step, and per 32 rows
// what its wavefront columns cost, idle ones among them, which is less where no window is padded).
inline double others_us(int64_t M, int64_t K, int64_t N, bool padded) {
  const int64_t tiles = (M + 31) / 32, cols = (N + 63) / 64;
  if (conv_streams(K, N, false, tiles * cols / 1024)) {
    const double per_rows = (cols == 1 ? 0.2 : cols == 2 ? 1.5 : cols <= 4 ? 6.1 : 26.0) * (padded ? 1.0 : 0.56);
    return 6.0 + static_cast<double>(tiles) / 4096 * (4.56 * static_cast<double>(cols) + per_rows);
  }
  const double steps = static_cast<double>((K + 63) / 64);
  auto rounds = [&](int bm, int bn) { return static_cast<double>((((M + bm - 1) / bm) * ((N + bn - 1) / bn) + 255) / 256); };
  switch (pick_conv_tile(M, N)) {
    case 0: return 1.7 + rounds(256, 128) * (5.8 + 0.66 * steps);
    case 1: return 4.1 + rounds(128, 128) * (1.4 + 0.324 * steps);
    default: return 3.7 + rounds(64, 64) * 0.15 * steps;
  }
}

}  // namespace itexhip
#endif  // ITEXHIP_QCONV_WALK_HPP_
