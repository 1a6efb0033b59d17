// Transpose of quantized tensors (_QuantizedTranspose: itex/core/kernels/common/transpose_op.h:197-236).
// Pure data movement, HBM-bound: 2 bytes of traffic per tensor byte.
#include <algorithm>

#include "qgemm_common.hpp"

namespace itexhip {
namespace {

constexpr int kMaxRank = 8;

struct TransposeArgs {
  int rank;                   // after merging
  int64_t out_dims[kMaxRank];
  int64_t in_stride[kMaxRank];  // stride in the input (in units) of output dimension i
  int64_t out_stride[kMaxRank];
  FastDiv by_dim[kMaxRank];     // small tensors: division by out_dims[i]
  int units;                    // small tensors: units per thread, 1 or 2
  int64_t total;              // number of units
};

// One unit (UNIT bytes) per thread and iteration: the output is written linearly, the input address
// comes from the output coordinates.
template <typename unit_t>
__global__ __launch_bounds__(256) void transpose_kernel(const TransposeArgs a, const unit_t* __restrict__ x,
                                                        unit_t* __restrict__ y) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t o = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; o < a.total; o += stride) {
    int64_t rem = o, src = 0;
#pragma unroll
    for (int d = kMaxRank - 1; d >= 0; --d) {
      if (d >= a.rank) continue;
      const int64_t q = d == 0 ? 0 : rem / a.out_dims[d];
      src += (rem - q * a.out_dims[d]) * a.in_stride[d];
      rem = q;
    }
    y[o] = x[src];
  }
}

// The same for fewer than 2^31 units (every index fits 32 bits): coordinates by multiply-shift divisions, UNITS loads of a
// thread in flight before it stores, and the dimensions walked in whichever of the two tensors' orders the host found
// better (see walk_order).  Bound by memory; three head splits and one merge of 128 x 128 x 12 x 64 bytes: 7.8 us each on average
// with 64-bit divisions in the output's order, 7.8 us with these divisions alone, 6.3 us with the order as well.
template <typename unit_t, int RANK, int UNITS>
__global__ __launch_bounds__(256) void transpose_small_kernel(const TransposeArgs a, const unit_t* __restrict__ x,
                                                              unit_t* __restrict__ y) {
  const uint32_t o0 = blockIdx.x * (256u * UNITS) + threadIdx.x, total = static_cast<uint32_t>(a.total);
  unit_t v[UNITS];
  uint32_t dst[UNITS];
#pragma unroll
  for (int u = 0; u < UNITS; ++u) {
    uint32_t rem = min(o0 + u * 256u, total - 1), src = 0;  // past the end: reads the last unit, stores nothing
    dst[u] = 0;
#pragma unroll
    for (int d = RANK - 1; d >= 0; --d) {
      if (d >= a.rank) continue;
      const uint32_t q = d == 0 ? 0 : static_cast<uint32_t>(fast_div(static_cast<int>(rem), a.by_dim[d]));
      const uint32_t i = rem - q * static_cast<uint32_t>(a.out_dims[d]);
      src += i * static_cast<uint32_t>(a.in_stride[d]);
      dst[u] += i * static_cast<uint32_t>(a.out_stride[d]);
      rem = q;
    }
    v[u] = x[src];
  }
#pragma unroll
  for (int u = 0; u < UNITS; ++u)
    if (o0 + u * 256u < total) y[dst[u]] = v[u];
}

template <typename unit_t>
void launch(const TransposeArgs& a, const void* x, void* y, hipStream_t st) {
  const unit_t* xp = static_cast<const unit_t*>(x);
  unit_t* yp = static_cast<unit_t*>(y);
  if (a.total < (1LL << 31)) {
    const unsigned blocks = static_cast<unsigned>((a.total + 256 * a.units - 1) / (256 * a.units));
    if (a.units == 1) {
      if (a.rank <= 4) transpose_small_kernel<unit_t, 4, 1><<<blocks, 256, 0, st>>>(a, xp, yp);
      else transpose_small_kernel<unit_t, kMaxRank, 1><<<blocks, 256, 0, st>>>(a, xp, yp);
    } else {
      if (a.rank <= 4) transpose_small_kernel<unit_t, 4, 2><<<blocks, 256, 0, st>>>(a, xp, yp);
      else transpose_small_kernel<unit_t, kMaxRank, 2><<<blocks, 256, 0, st>>>(a, xp, yp);
    }
    return;
  }
  const int64_t blocks = std::min<int64_t>((a.total + 255) / 256, 256 * 16);
  transpose_kernel<unit_t><<<static_cast<unsigned>(blocks), 256, 0, st>>>(a, xp, yp);
}

// How many 128-byte lines of the other tensor a walk fetches (or writes back) per unit, where `cache` bytes of them stay close:
// the walk's dimensions, innermost first, make a window of units whose lines just fit; beyond it every line comes again.
struct WalkDim {
  int64_t extent, stride;  // stride in the other tensor, in units
};
double lines_per_unit(const WalkDim* walk, int n, int unit, double cache) {
  double units = 1.0, rows = 1.0, span = unit;  // of the window: rows of `span` bytes each
  for (int i = 0; i < n; ++i) {
    const double extent = static_cast<double>(walk[i].extent), step = static_cast<double>(walk[i].stride) * unit;
    const bool near = step < 128.0;  // neighbours along this dimension share lines
    const double lines = rows * std::max(1.0, span / 128.0);
    const double whole = near ? rows * std::max(1.0, (span + (extent - 1.0) * step) / 128.0) : lines * extent;
    if (whole * 128.0 > cache) {  // a part of this dimension fills the window
      const double part = std::max(1.0, std::min(extent, near ? extent * cache / (whole * 128.0) : cache / (lines * 128.0)));
      return (near ? rows * std::max(1.0, (span + (part - 1.0) * step) / 128.0) : lines * part) / (units * part);
    }
    units *= extent;
    if (near) span += (extent - 1.0) * step;
    else rows *= extent;
  }
  return rows * std::max(1.0, span / 128.0) / units;
}

// Order and units per thread of a small tensor.  One tensor is walked from end to end, the other one jumps: the order is that of
// the output unless the input's brings the jumping tensor through an L2 (4 MB of lines) at most half as often, or, where neither
// does in 8 MB and more, needs at most two thirds of the lines within 8 KB, what two wavefronts have in flight.  Single units
// whose neighbours go out a multiple of 4 KB apart meet in the same sets and channels and stay in the output's order (3 x 64 x
// 768 x 256 bytes (3, 1, 2, 0) 164 us, input's 552).  Two units per thread overlap two loads; one leaves more threads, and more
// lines close by where the rows of the input are lines of their own.
// us, one unit per thread in the output's / the input's order: 36 x 50 x 246 x 16 ints (3, 0, 1, 2) 68.3 / 19.4, 44 x 167 x 306
// x 5 (2, 1, 3, 0) 48 / 146, 54 x 284 x 122 x 16 (2, 1, 3, 0) 197 / 365, 267 x 133 x 24 x 64 bytes (3, 2, 0, 1) 969 / 251; the
// head split of 128 x 128 x 12 x 64 bytes 7.8 / 6.3 (the second rule).  Over 15000 shapes of up to 5 dimensions and 64 MB the
// choice is 3 % above the fastest of the four, 5 % over 7600 whose extents are powers of two and three times such; rules on the
// two innermost dimensions alone were 5.4 and 5.8 % above it.  1.6 and 2.5 % of them take longer than in the output's order
// with threads that return for more and 64-bit divisions (51 x 680 x 320 bytes reversed 65 us, here 150): both tensors jump by
// whole lines there.
// us, one / two units: 300 x 301 x 302 bytes reversed 338 / 205, 1024 x 1024 4.8 / 5.9, 1024 x 4096 x 16 (1, 0, 2) 30.6 / 49.9.
void walk_order(TransposeArgs& a, int unit) {
  int n = a.rank;
  const bool in_runs = a.in_stride[n - 1] == 1 && a.out_dims[n - 1] > 1;
  if (n > 1 && a.out_dims[n - 1] == 1) a.rank = --n;  // one unit: no dimension of its own
  int order[kMaxRank];
  for (int i = 0; i < n; ++i) order[i] = i;
  std::sort(order, order + n, [&](int p, int q) { return a.in_stride[p] > a.in_stride[q]; });
  const double bytes = static_cast<double>(a.total) * unit, mb = 1024.0 * 1024.0;
  WalkDim out[kMaxRank], in[kMaxRank];
  for (int i = 0; i < n; ++i) {
    const int o = n - 1 - i, p = order[n - 1 - i];
    out[i] = WalkDim{a.out_dims[o], a.in_stride[o]};
    in[i] = WalkDim{a.out_dims[p], a.out_stride[p]};
  }
  const double l2_out = lines_per_unit(out, n, unit, 4.0 * mb), l2_in = lines_per_unit(in, n, unit, 4.0 * mb);
  bool by_input = 2.0 * l2_in < l2_out;
  if (!by_input && 2.0 * l2_out >= l2_in && bytes >= 8.0 * mb)
    by_input = 1.5 * lines_per_unit(in, n, unit, 8192.0) < lines_per_unit(out, n, unit, 8192.0);
  if (by_input && !in_runs) {
    int i = 0;
    while (i < n && in[i].stride * unit < 128) ++i;
    if (i < n && in[i].extent >= 8 && in[i].stride * unit % 4096 == 0) by_input = false;
  }
  const bool own_lines = unit == 16 && !in_runs && a.out_dims[order[n - 1]] % 8 == 0;  // rows of whole lines
  a.units = bytes <= (unit == 1 ? (in_runs ? 0.25 : 1.0) : unit == 4 && in_runs ? 1.0 : 8.0) * mb || own_lines ? 1 : 2;
  if (!by_input) return;
  const TransposeArgs b = a;
  for (int i = 0; i < n; ++i) {
    a.out_dims[i] = b.out_dims[order[i]];
    a.in_stride[i] = b.in_stride[order[i]];
    a.out_stride[i] = b.out_stride[order[i]];
  }
}

}  // namespace
}  // namespace itexhip

using namespace itexhip;

extern "C" int itexhip_transpose(const void* x, void* y, int elem_size, int rank, const int64_t* dims, const int32_t* perm,
                                 void* stream) {
  const char* who = "itexhip_transpose";
  ITEXHIP_REQUIRE(elem_size == 1 || elem_size == 4, "%s: element size %d (1 or 4)", who, elem_size);
  ITEXHIP_REQUIRE(rank >= 0 && rank <= kMaxRank, "%s: rank %d (at most %d)", who, rank, kMaxRank);
  ITEXHIP_REQUIRE(rank == 0 || (dims && perm), "%s: null dims or perm", who);
  bool seen[kMaxRank] = {false};
  int64_t total = 1;
  for (int i = 0; i < rank; ++i) {
    ITEXHIP_REQUIRE(perm[i] >= 0 && perm[i] < rank && !seen[perm[i]], "%s: perm is not a permutation", who);
    seen[perm[i]] = true;
    ITEXHIP_REQUIRE(dims[i] >= 0, "%s: negative dimension", who);
    total *= dims[i];
  }
  if (total == 0) return ITEXHIP_OK;
  ITEXHIP_REQUIRE(x && y && aligned(x, elem_size) && aligned(y, elem_size), "%s: null or misaligned buffer", who);

  // input strides (elements), then the output's view of them; dimensions of extent 1 drop out
  int64_t in_stride[kMaxRank], od[kMaxRank], os[kMaxRank];
  {
    int64_t st = 1;
    for (int i = rank - 1; i >= 0; --i) { in_stride[i] = st; st *= dims[i]; }
  }
  int n = 0;
  for (int i = 0; i < rank; ++i) {
    if (dims[perm[i]] == 1) continue;
    od[n] = dims[perm[i]];
    os[n] = in_stride[perm[i]];
    // merge with the previous output dimension when the two are also adjacent, in this order, in the input
    if (n > 0 && os[n - 1] == os[n] * od[n]) {
      od[n - 1] *= od[n];
      os[n - 1] = os[n];
    } else {
      ++n;
    }
  }
  if (n == 0) { od[0] = 1; os[0] = 1; n = 1; }  // a single element

  // the innermost run: contiguous in both tensors when its input stride is 1
  int64_t bytes_inner = os[n - 1] == 1 ? od[n - 1] * elem_size : 0;
  int unit = elem_size;
  if (bytes_inner >= 16 && bytes_inner % 16 == 0 && aligned(x, 16) && aligned(y, 16)) {
    bool ok = true;  // every other stride must keep 16-byte alignment
    for (int i = 0; i + 1 < n; ++i) ok = ok && (os[i] * elem_size) % 16 == 0;
    if (ok) unit = 16;
  } else if (elem_size == 1 && bytes_inner >= 4 && bytes_inner % 4 == 0 && aligned(x, 4) && aligned(y, 4)) {
    bool ok = true;
    for (int i = 0; i + 1 < n; ++i) ok = ok && os[i] % 4 == 0;
    if (ok) unit = 4;
  }
  const int per = unit / elem_size;  // elements per unit
  TransposeArgs a{};
  a.rank = n;
  for (int i = 0; i < n; ++i) {
    a.out_dims[i] = od[i];
    a.in_stride[i] = os[i] / (i + 1 < n ? per : 1);
  }
  if (per > 1) { a.out_dims[n - 1] = od[n - 1] / per; a.in_stride[n - 1] = 1; }
  a.total = total / per;
  if (a.total < (1LL << 31)) {
    int64_t s = 1;
    for (int i = n - 1; i >= 0; --i) { a.out_stride[i] = s; s *= a.out_dims[i]; }
    walk_order(a, unit);
    for (int i = 0; i < a.rank; ++i) a.by_dim[i] = make_fast_div(a.out_dims[i]);
  }
  hipStream_t st = as_stream(stream);
  if (unit == 16) launch<i4>(a, x, y, st);
  else if (unit == 4) launch<uint32_t>(a, x, y, st);
  else launch<uint8_t>(a, x, y, st);
  ITEXHIP_CHECK_LAUNCH(who);
  return ITEXHIP_OK;
}
