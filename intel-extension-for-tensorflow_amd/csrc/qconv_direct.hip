// Quantized 3 x 3 Conv2D of stride 1 with 32 to 128 input channels and an 8-bit result: the middle convolution of a residual
// block.  As an implicit GEMM on tiles it loads every input byte nine times into LDS and the weight once per tile, waits at a
// barrier per 64-deep K step, and its address arithmetic and sign flips stand between the MFMAs.
//
// Here a workgroup takes a run of 32-row tiles of the result and puts the input rows that their windows touch into LDS once,
// padding included and sign flipped; the images are treated as lying one below the other, each with its padding, so that the
// run may cross from one to the next.  A wavefront keeps the weight of its 32 channels in registers (36 per 32 input
// channels) and walks the tiles without another barrier: a fragment read of 16 bytes per lane and an MFMA per 32-deep
// chunk, the fragments 6 or 9 chunks ahead of their use and over the border between two tiles.  Pixels lie an odd number of 16-byte
// pieces apart in LDS, so that the reads of 16 neighbours fall into different banks.  As in qgemm_stream.hip a lane ends with
// 16 consecutive channels of one position, packed in registers.
//
// Tile kernel -> this one, us: 32 x 56 x 56 x 64 -> 64 12.4 -> 8.0, 32 x 28 x 28 x 128 -> 128 10.9 -> 7.9, 32 x 25 x 25 x 128 -> 128
// 10.7 -> 7.0, 64 x 56 x 56 x 64 -> 64 19.9 -> 12.6, 32 x 112 x 112 x 64 -> 64 35.4 -> 24.4, 32 x 56 x 56 x 96 -> 96 29.7 -> 16.6, one
// 32 x 32 x 64 -> 128 5.5 -> 4.0; the kernel for a short K -> this one: 32 x 112 x 112 x 32 -> 32 18.6 -> 10.0.  What bounds it:
// the start of a launch (3.7: input rows and weight on their way, together), then a wavefront's tile after another, MFMAs
// (18 of 32 cycles with 64 channels) and epilogue in turn.  Fragments two chunks ahead left every pair of MFMAs waiting for LDS (0.25 of
// 1.0 us per tile with 128 channels); row addresses in scalar arithmetic, a branch per piece, were 0.3 slower than the counters.
#include "qconv_walk.hpp"
#include "qgemm_pack.hpp"

namespace itexhip {
namespace {

constexpr int kForceDirect = 17;  // of itexhip_test_force_tile_shape

struct DirectArgs : DirectGeometry<FastDiv> {
  int N;
  int waves_n;        // wavefronts side by side along the channels: 1, 2 or 4
  int wgs;            // workgroups with tiles
  int panel;          // offset of the channel parameters in LDS
  float lo, hi;       // post-op bounds, see POST
  const int32_t* colsum;
  const float *scales, *bias;
  int comp_mul, n_scales;
};

// Registers: 126 with 32 channels, four wavefronts per SIMD; 152 with 64 (72 of weight), three; 200 and 224 (144 of weight), two.
template <int OUT_T, int POST, int C32>
__global__ __launch_bounds__(256, C32 == 1 ? 4 : C32 == 2 ? 3 : 2) void qconv_direct_kernel(
    const uint8_t* __restrict__ a, uint32_t amask, const uint8_t* __restrict__ bp, const DirectArgs s,
    uint8_t* __restrict__ out) {
  constexpr int CHUNKS = 9 * C32, PIECES = 2 * C32;  // 32-deep K chunks; 16-byte pieces of a pixel
  constexpr int PITCH = PIECES * 16 + 16;            // of a pixel in LDS: an odd number of pieces
  constexpr int BATCH = 8;
  constexpr int AHEAD = C32 % 2 != 0 ? 9 : 6;         // fragments on their way from LDS
  static_assert(CHUNKS % AHEAD == 0, "the ring of fragments closes over a tile");
  extern __shared__ __align__(16) uint8_t lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lrow = lane & 31, half = lane >> 5;
  const int wn = wave % s.waves_n, wm = wave / s.waves_n, waves_m = 4 / s.waves_n;
  const int channels = s.waves_n * 32, n_base = blockIdx.y * channels, n0 = n_base + wn * 32;
  // consecutive workgroup ids go round the 8 XCDs: each of them takes a contiguous range of rows
  const int wg = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (wg >= s.wgs) return;
  const int t0 = wg * s.per_wg, t1 = min(t0 + s.per_wg, s.tiles);

  const int v0 = s.first_row(t0), v1 = s.last_row(t1);
  // ---- the channel parameters, the input rows and the weight travel together
  const int channel = n_base + min(static_cast<int>(threadIdx.x), channels - 1);
  const int colsum = s.colsum ? s.colsum[channel] : 0;
  const float scale = s.n_scales > 0 ? s.scales[s.n_scales > 1 ? channel : 0] : 1.0f;
  const float bias = s.bias[channel];

  const int pieces = (v1 - v0) * s.wp * PIECES, row_bytes = s.wp * PITCH;
  InputWalk<PIECES, FastDiv> walk(s, v0, static_cast<int>(threadIdx.x));
  auto fetch = [&](int i) -> v4i {  // what is outside reads 16 zero bytes
    uint32_t offset;
    const bool inside = walk.inside(s, &offset) & (i < pieces);
    const uint8_t* src = a + offset;  // (before the choice: a branch per piece otherwise)
    src = inside ? src : reinterpret_cast<const uint8_t*>(kZeros);
    walk.advance(s);
    return *reinterpret_cast<const v4i*>(src);
  };
  auto put = [&](int i, v4i x) {
    x.x ^= amask; x.y ^= amask; x.z ^= amask; x.w ^= amask;
    if (i < pieces) *reinterpret_cast<v4i*>(lds + piece_at<PIECES>(i)) = x;
  };
  const int t = threadIdx.x;
  v4i x[BATCH];
#pragma unroll
  for (int u = 0; u < BATCH; ++u) x[u] = fetch(t + u * 256);
  v4i w[CHUNKS];
  {
    const int ch = ((lrow >> 2) & 1) * 16 + (lrow >> 3) * 4 + (lrow & 3);
    const uint8_t* src = bp + static_cast<int64_t>(n0 >> 5) * (2 * ((CHUNKS + 1) / 2)) * kChunkBytes;
    const uint32_t off = static_cast<uint32_t>((lane & 32) + ch) * 16u;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) w[c] = *reinterpret_cast<const v4i*>(src + c * kChunkBytes + off);
  }
  int* const p_comp = reinterpret_cast<int*>(lds + s.panel);
  float* const p_scale = reinterpret_cast<float*>(p_comp + channels);
  float* const p_bias = p_scale + channels;
  if (static_cast<int>(threadIdx.x) < channels) {
    p_comp[threadIdx.x] = s.comp_mul * colsum;
    p_scale[threadIdx.x] = scale;
    p_bias[threadIdx.x] = bias;
  }
#pragma unroll
  for (int u = 0; u < BATCH; ++u) put(t + u * 256, x[u]);
  for (int i0 = BATCH * 256; i0 < pieces; i0 += BATCH * 256) {
#pragma unroll
    for (int u = 0; u < BATCH; ++u) x[u] = fetch(i0 + t + u * 256);
#pragma unroll
    for (int u = 0; u < BATCH; ++u) put(i0 + t + u * 256, x[u]);
  }
  __syncthreads();

  if (t0 + wm >= t1) return;  // whole wavefront; no barrier follows
  const int channel_off = half * 16;
  auto origin_of = [&](int tile) -> const uint8_t* {  // of the window of the lane's output position
    return lds + s.window_at(min(tile * 32 + lrow, s.M - 1), v0, row_bytes, PITCH) + channel_off;
  };
  auto fragment = [&](const uint8_t* origin, auto c) -> v4i {
    constexpr int k = decltype(c)::value / C32, kh = k / 3, kw = k % 3;
    return *reinterpret_cast<const v4i*>(origin + kh * row_bytes + (kw * PITCH + decltype(c)::value % C32 * 32));
  };
  v4i f[AHEAD];
  const uint8_t* origin = origin_of(t0 + wm);
  static_for<AHEAD>([&](auto c) { f[c] = fragment(origin, c); });
  for (int tile = t0 + wm; tile < t1; tile += waves_m) {
    const uint8_t* const next = origin_of(tile + waves_m < t1 ? tile + waves_m : tile);
    int col0 = wn * 32 + half * 16;
    asm volatile("" : "+v"(col0));
    v16i acc;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const v4i c = *reinterpret_cast<const v4i*>(p_comp + col0 + q * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[q * 4 + r] = c[r];
    }
    static_for<CHUNKS>([&](auto c) {
      constexpr int ci = decltype(c)::value, ahead = ci + AHEAD;
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[ci], f[ci % AHEAD], acc, 0, 0, 0);
      f[ci % AHEAD] = fragment(ahead < CHUNKS ? origin : next, std::integral_constant<int, ahead % CHUNKS>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    origin = next;
    const int m = tile * 32 + lrow;
    v4i packed;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f4 sc = *reinterpret_cast<const f4*>(p_scale + col0 + q * 4);
      const f4 bi = *reinterpret_cast<const f4*>(p_bias + col0 + q * 4);
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = static_cast<float>(acc[q * 4 + r]) * sc[r];
        v[r] = v[r] + bi[r];
        if constexpr (POST == kPostRelu && OUT_T != ITEXHIP_QUINT8) v[r] = fmaxf(v[r], 0.0f);
        if constexpr (POST == kPostClip) v[r] = __builtin_amdgcn_fmed3f(v[r], s.lo, s.hi);  // lo <= hi; lo for NaN, as min(max()) gives
      }
      packed[q] = static_cast<int>(pack_bytes<OUT_T, POST>(v));
    }
    if (m < s.M)
      *reinterpret_cast<v4i*>(out + (static_cast<uint32_t>(m) * static_cast<uint32_t>(s.N) + static_cast<uint32_t>(n0 + half * 16))) = packed;
  }
}

template <int OUT_T, int POST, int C32>
int launch(const uint8_t* a, uint32_t amask, const uint8_t* bp, const DirectArgs& s, uint8_t* out, dim3 grid, size_t lds, hipStream_t st) {
  auto kern = qconv_direct_kernel<OUT_T, POST, C32>;
  static unsigned long long attr_done = 0;  // devices on which this instantiation's attribute is set
  if (!device_bit(&attr_done, false)) {
    hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsPerCu);
    if (err != hipSuccess) return hip_fail(err, "hipFuncSetAttribute(qconv_direct_kernel)");
    device_bit(&attr_done, true);
  }
  note_kernel(kLastDirect, s.per_wg);
  kern<<<grid, 256, lds, st>>>(a, amask, bp, s, out);
  return ITEXHIP_OK;
}

template <int OUT_T, int C32>
int dispatch(const uint8_t* a, uint32_t amask, const uint8_t* bp, const DirectArgs& s, int post, uint8_t* out,
             dim3 grid, size_t lds, hipStream_t st) {
  switch (post) {
    case kPostNone: return launch<OUT_T, kPostNone, C32>(a, amask, bp, s, out, grid, lds, st);
    case kPostRelu: return launch<OUT_T, kPostRelu, C32>(a, amask, bp, s, out, grid, lds, st);
    default: return launch<OUT_T, kPostClip, C32>(a, amask, bp, s, out, grid, lds, st);
  }
}

}  // namespace

// 1: the call was launched here; 0: not a call for this kernel; < 0: an error (the status, negated).
int try_direct(const uint8_t* a, uint32_t amask, const uint8_t* bp, int M, int K, int N, const EpilogueArgs& e, int out_type,
               void* out, hipStream_t st, const ConvTileArgs& cv) {
  if (out_type != ITEXHIP_QUINT8 && out_type != ITEXHIP_QINT8) return 0;
  const int forced = __atomic_load_n(&g_forced_tile_shape[1], __ATOMIC_RELAXED);  // tests ask for another kernel, or for this one
  if (forced >= 0 && forced != kForceDirect) return 0;
  if (cv.k_w != 3 || K != 9 * cv.in_c || cv.in_c % 32 != 0 || cv.in_c > 128 || cv.dil_h != 1 || cv.dil_w != 1 || cv.stride_h != 1 ||
      cv.stride_w != 1 || N % 32 != 0 || e.bias == nullptr || e.fused || e.addend || e.row_min_a)
    return 0;
  if (static_cast<int64_t>(M) * N >= (1LL << 31)) return 0;
  CanonChain c;
  const int act = canon_chain(e, &c);
  if (act < 0 || act > 2 || (c.flags & ~(kChainMax0 | kChainClip)) != 0) return 0;
  if ((c.flags & kChainClip) && !(c.lo <= c.hi)) return 0;  // the median of three is no clip then
  const int64_t wp = cv.out_w + 2LL, vr = cv.out_h + 2LL;
  if (wp * direct_pitch(cv.in_c) * 3 > kLdsPerCu || M / cv.out_w / cv.out_h * vr >= (1LL << 31)) return 0;
  const DirectPlan plan = plan_direct(M, cv.in_c, N, cv.out_h, cv.out_w);
  if (plan.per_wg == 0 || plan.groups_n > 65535) return 0;  // rows too wide for LDS; gridDim.y
  // Where it is the faster kernel.  What it loses to is the input it puts into LDS: rows of which a run needs several times its own
  // (11 x 253 x 253 x 32 -> 96 53 us, 75 here), and channels in many groups of which each puts the input there again (4 x 89 x 89 x
  // 96 -> 384 20.0, 29.8 here).  Both estimates follow it: over 3500 drawn shapes of 4 x 4 to 300 x 300 with 32 to 512 results
  // 0.745 of the other kernels' time in the mean, 12 of them more than 5 % longer, 1.16 at most.
  if (forced != kForceDirect && plan.us >= others_us(M, K, N, cv.pad_top > 0 || cv.pad_left > 0)) return 0;
  DirectArgs s{};
  s.M = M; s.N = N;
  s.in_h = cv.in_h; s.in_w = cv.in_w; s.out_h = cv.out_h; s.out_w = cv.out_w;
  s.pad_top = cv.pad_top; s.pad_left = cv.pad_left;
  s.by_out_w = cv.by_out_w; s.by_out_h = cv.by_out_h;
  set_walk(s, cv.in_c / 16, make_fast_div);
  s.tiles = static_cast<int>((static_cast<int64_t>(M) + 31) / 32);
  s.per_wg = plan.per_wg; s.wgs = plan.wgs; s.waves_n = plan.waves_n; s.panel = plan.panel;
  s.colsum = e.colsum; s.scales = e.scales; s.bias = static_cast<const float*>(e.bias);
  s.comp_mul = e.comp_mul; s.n_scales = e.n_scales;
  s.lo = c.lo; s.hi = c.hi;
  const int64_t lds = plan.lds;
  const dim3 grid(static_cast<unsigned>((s.wgs + 7) / 8 * 8), static_cast<unsigned>(plan.groups_n));
  const int post = c.flags & kChainClip ? kPostClip : c.flags & kChainMax0 ? kPostRelu : kPostNone;
  uint8_t* o = static_cast<uint8_t*>(out);
  int rc;
#define DIRECT(C32)                                                                                                       \
  rc = out_type == ITEXHIP_QUINT8 ? dispatch<ITEXHIP_QUINT8, C32>(a, amask, bp, s, post, o, grid, static_cast<size_t>(lds), st)             \
                                  : dispatch<ITEXHIP_QINT8, C32>(a, amask, bp, s, post, o, grid, static_cast<size_t>(lds), st)
  switch (cv.in_c / 32) {
    case 1: DIRECT(1); break;
    case 2: DIRECT(2); break;
    case 3: DIRECT(3); break;
    default: DIRECT(4); break;
  }
#undef DIRECT
  return rc == ITEXHIP_OK ? 1 : -rc;
}

}  // namespace itexhip
