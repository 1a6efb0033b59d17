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

// Order and units per thread of a small tensor.  Both tensors are walked in runs: the innermost dimension where it is
// contiguous in both, else single units.  Next to the run the output has a dimension of r, the input one of c.
// Runs of 4 units and more (64 bytes of a 16-byte unit): in the input's order where c < r (the head split: c = 12 heads, r =
// 128 tokens): a workgroup reads whole lines and writes runs of r instead of touching every line of the input once per head;
// two units per thread (1000 x 32 x 64 bytes, 32 of them: 24.5 us one unit, output's order; 21.2).
// Shorter runs: the same, where c is at most half of r, the r destinations of a workgroup's reads are worth a line (c * run
// up to 64) or do not lie a power of two apart; one unit per thread (its neighbours' units are other lines), or two where the
// rows of the input share lines.  us, output's / input's order: 1000 x 32 x 16 bytes 11.7 / 6.7, 1000 x 7 x 600 x 16 74 / 58,
// 4096 x 256 x 16 8.4 / 17.6, 4096 x 1024 x 16 22.8 / 39.9, 12 x 197 x 16 2.4 / 3.1; one / two units: 1024 x 1024 x 16 9.6 /
// 15.0, 1024 x 4096 x 16 30.6 / 49.9, 300 x 301 x 16 52.7 / 42.7.
// Bytes: always two but for small tensors (300 x 301 x 302 reversed 205 us, one unit 338; 1024 x 1024 5.9, one unit 4.8).
void walk_order(TransposeArgs& a, int unit) {
  int n = a.rank;
  const bool in_runs = a.in_stride[n - 1] == 1 && a.out_dims[n - 1] > 1;
  if (n > 1 && a.out_dims[n - 1] == 1) a.rank = --n;  // one unit: no dimension of its own
  int order[kMaxRank];
  for (int i = 0; i < n; ++i) order[i] = i;
  std::sort(order, order + n, [&](int p, int q) { return a.in_stride[p] > a.in_stride[q]; });
  bool by_input = false;
  a.units = 2;
  const int next = in_runs ? n - 2 : n - 1;
  if (next >= 0) {
    const int64_t run = in_runs ? a.out_dims[n - 1] : 1, r = a.out_dims[next], c = a.out_dims[order[next]];
    if (in_runs && (run >= 4 || unit == 1)) {
      by_input = c < r;
    } else if (unit > 1) {
      by_input = 2 * c <= r && r >= 32 && (c * run <= 64 || (r * run * unit) % 4096 != 0);
      a.units = unit == 16 && !by_input && (c * run * unit) % 128 != 0 ? 2 : 1;
    } else if (a.total <= 1 << 20) {
      a.units = 1;
    }
  }
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
