// Quantized MatMul and Conv2D with a short K, many rows and an 8-bit result: the 1 x 1 and first convolutions of vision
// networks, pointwise convolutions, narrow linears.  Such a launch is bound by the bytes of its activations, result and
// residual, and by the instructions of its epilogue; the tile kernel spends it on three K steps of loads that a K of 64
// does not have, on barriers and on a transposition of the result through LDS.
//
// Here the weight of a workgroup's channels (K x 64 per wavefront column) and their parameters are put into LDS once, and
// the wavefronts then walk the rows without another barrier.  A wavefront takes 32 rows x 64 channels at a time: its
// activation fragments come straight from global memory (a lane loads 16 consecutive k of one row; a convolution resolves
// the window position per 16-byte piece), a group of them ahead of the MFMAs that use them.  The weight is the first MFMA
// operand and its channels are put into LDS in an order that leaves a lane with 16 consecutive channels of one row: the
// result is packed in registers and goes out as 16-byte stores, and a residual comes in as 16-byte loads a tile ahead.
//
// Measured, tile kernel -> this one, us: 401408 x 32 -> 64 with a clip 18.4 -> 9.9; 100352 x 64 -> 256 with a residual and
// a ReLU 24.3 -> 14.4; 7 x 7 convolution over 32 x 224 x 224, stride 2, 224 bytes of patch -> 64 channels 30.1 -> 12.8.
// What bounds it there: the start of a launch that fills the device (parameters and weight on their way to LDS, first rows,
// last stores: 5 us), then vector instructions (6 per result with a clip, 7 with a residual) and the results leaving L2
// (401408 x 32 -> 64: 5 us beyond the start, 7.7 TB/s).
#include "qconv_walk.hpp"
#include "qgemm_pack.hpp"

namespace itexhip {
namespace {

constexpr int kMaxWeightBytes = 72 * 1024;  // of a workgroup: two of them per CU
constexpr int kForceStream = 16;            // of itexhip_test_force_tile_shape
constexpr int kBlocks = 2;                  // 32-channel blocks per wavefront (the stores are laid out for two)

struct StreamArgs {
  int M, K, N;
  int chunks;       // 32-deep K chunks that hold data
  int packed_kt;    // K chunks of the packed weight (K padded to a multiple of 64)
  FastDiv by_chunks;
  int waves_n;      // wavefronts side by side along N: 1, 2 or 4
  int tiles;        // row tiles of 32
  int walkers;      // wavefronts that share them (per wavefront column)
  uint64_t share;   // 2^24 * tiles / walkers: wavefront w takes the tiles from (w * share) >> 24 on
  int padded;       // convolution: a window may reach into the padding
  float lo, hi;     // post-op bounds, see POST
  float sum_scale;
};

// 128 vector registers for four wavefronts per SIMD, without scratch but for groups of 4 with a residual (it costs a launch
// 1.5 us); up to 26 scalar registers go to lanes of a vector register.
// HOLD: the K chunks of a tile are exactly GROUP; all are held at once, and each is replaced by the next tile's as soon as its
// MFMAs are issued: no second set of registers, no copies, and where a lane's pieces lie relative to its row is computed
// once.  With two sets, copies and 21 instructions per piece the 7 x 7 convolution above took 14.6 us and 401408 x 32 -> 64
// with a clip 10.9.  Otherwise GROUP chunks are multiplied while the next GROUP travel.
template <int OUT_T, int POST, int SUM, int GROUP, bool CONV, bool HOLD>
__global__ __launch_bounds__(256, 4) void qgemm_stream_kernel(const uint8_t* __restrict__ a, uint32_t amask,
                                                            const uint8_t* __restrict__ bp, const StreamArgs s, EpilogueArgs e,
                                                            uint8_t* __restrict__ out, const ConvTileArgs cv) {
  extern __shared__ __align__(16) uint8_t lds[];  // [waves_n * kBlocks][chunks] fragments, parameters, window table
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lrow = lane & 31, half = lane >> 5;
  const int channels = s.waves_n * kBlocks * 32;            // of this workgroup
  const int n_base = blockIdx.y * channels;
  const int frags = s.waves_n * kBlocks * s.chunks;
  int* const p_comp = reinterpret_cast<int*>(lds + frags * kChunkBytes);
  float* const p_scale = reinterpret_cast<float*>(p_comp + channels);
  float* const p_bias = p_scale + channels;
  int2* const table = reinterpret_cast<int2*>(p_bias + channels);  // convolution, not HOLD: per 16-byte piece of a patch row

  const int wn = wave % s.waves_n, wm = wave / s.waves_n, waves_m = 4 / s.waves_n;
  // consecutive workgroup ids go round the 8 XCDs: each of them walks a contiguous range of rows (neighbouring rows of a
  // convolution read the same input); gridDim.x is a multiple of 8
  const int wg = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int walker = wg * waves_m + wm;
  const int t0 = static_cast<int>((walker * s.share) >> 24);
  const int t1 = walker >= s.walkers ? 0 : walker + 1 == s.walkers ? s.tiles : static_cast<int>(((walker + 1) * s.share) >> 24);
  const int klast = s.K - 16, plast = (s.K >> 4) - 1;

  // ---- where the lane's row of a tile begins
  uint32_t row_off;
  int win_h = 0, win_w = 0;
  auto locate = [&](int tile) {
    const int m = min(tile * 32 + lrow, s.M - 1);
    if constexpr (CONV) {
      const int t = fast_div(m, cv.by_out_w), ow = m - t * cv.out_w;
      const int b = fast_div(t, cv.by_out_h), oh = t - b * cv.out_h;
      win_h = oh * cv.stride_h - cv.pad_top;
      win_w = ow * cv.stride_w - cv.pad_left;
      row_off = static_cast<uint32_t>(((b * cv.in_h + win_h) * cv.in_w + win_w) * cv.in_c);
    } else {
      row_off = static_cast<uint32_t>(m) * static_cast<uint32_t>(s.K);  // M * K < 2^31 checked by the host
    }
  };
  auto window_piece = [&](int p) {  // {window row << 16 | window column, byte offset from the window's origin}
    const int k0 = p * 16;
    const int kk = fast_div(k0, cv.by_in_c), cc = k0 - kk * cv.in_c;
    const int kh = fast_div(kk, cv.by_k_w), kw = kk - kh * cv.k_w;
    const int dh = kh * cv.dil_h, dw = kw * cv.dil_w;  // < 2^15 each, checked by the host
    return make_int2((dh << 16) | dw, (dh * cv.in_w + dw) * cv.in_c + cc);
  };
  auto load_piece = [&](const int2 piece) -> v4i {
    const uint8_t* src = a + (row_off + static_cast<uint32_t>(piece.y));
    if (s.padded) {  // a position in the padding reads 16 zero bytes
      const int ih = win_h + (piece.x >> 16), iw = win_w + (piece.x & 0xffff);
      const bool inside = static_cast<unsigned>(ih) < static_cast<unsigned>(cv.in_h) &&
                          static_cast<unsigned>(iw) < static_cast<unsigned>(cv.in_w);
      src = inside ? src : reinterpret_cast<const uint8_t*>(kZeros);
    }
    return *reinterpret_cast<const v4i*>(src);
  };
  // fragment of chunk c: k beyond K meets zero weights, any bytes of the tensor will do there
  auto load = [&](int c) -> v4i {
    if constexpr (CONV) return load_piece(table[min(c * 2 + half, plast)]);
    else return *reinterpret_cast<const v4i*>(a + (row_off + static_cast<uint32_t>(min(c * 32 + half * 16, klast))));
  };

  // (convolution: lane p works out piece p, the others read it from there; GROUP <= 8 of 2 pieces)
  int2 mine = make_int2(0, 0);
  if constexpr (CONV) mine = window_piece(min(lane, plast));
  auto piece_of = [&](int c) {
    const int p = min(c * 2 + half, plast);
    return make_int2(__shfl(mine.x, p, 64), __shfl(mine.y, p, 64));
  };
  uint32_t offset[HOLD ? GROUP : 1];  // HOLD: of the lane's piece of chunk u, from the beginning of its row
  if constexpr (HOLD) {
#pragma unroll
    for (int u = 0; u < GROUP; ++u) {
      if constexpr (CONV) offset[u] = static_cast<uint32_t>(piece_of(u).y);
      else offset[u] = static_cast<uint32_t>(min(u * 32 + half * 16, klast));
    }
  }
  auto load_held = [&](int u) -> v4i { return *reinterpret_cast<const v4i*>(a + (row_off + offset[u])); };

  // ---- the first fragments travel while the weight is put into LDS (without the window table, which is not there yet)
  v4i cur[GROUP], nxt[HOLD ? 1 : GROUP];
  locate(t0);  // (a wavefront without rows reads the last row)
#pragma unroll
  for (int u = 0; u < GROUP; ++u) {
    const int c = min(u, s.chunks - 1);
    if constexpr (HOLD) cur[u] = load_held(u);
    else if constexpr (CONV) cur[u] = load_piece(piece_of(c));
    else cur[u] = load(c);
  }

  // the residual of a tile: 16 consecutive channels per block of the lane's row
  typedef int v4i_a4 __attribute__((ext_vector_type(4), aligned(4)));
  const int n0 = n_base + wn * (kBlocks * 32);
  v4i add[kBlocks], add_nxt[kBlocks];
  auto load_add = [&](int tile, v4i (&d)[kBlocks]) {
    if constexpr (SUM != 0) {
      const uint32_t o = static_cast<uint32_t>(min(tile * 32 + lrow, s.M - 1)) * static_cast<uint32_t>(s.N);
#pragma unroll
      for (int b = 0; b < kBlocks; ++b)  // (channels past N: the row's last 16, not used)
        d[b] = *reinterpret_cast<const v4i_a4*>(static_cast<const uint8_t*>(e.addend) + (o + min(n0 + b * 32 + half * 16, s.N - 16)));
    }
  };
  load_add(t0, add);

  // ---- the weight: row r of a fragment holds channel (r / 4 % 2) * 16 + (r / 8) * 4 + r % 4 of its block, so that the 16
  // results of a lane (rows (i / 4) * 8 + half * 4 + i % 4) are channels half * 16 .. half * 16 + 15.  Direct global -> LDS
  // loads (lane l's 16 bytes land at 16 l): all of them are in flight at once, where a loop over registers waits for each.
  {
    const int ch = ((lrow >> 2) & 1) * 16 + (lrow >> 3) * 4 + (lrow & 3);
    const int last_nt = ((s.N + 31) >> 5) - 1;
    for (int f = wave; f < frags; f += 4) {
      const int block = fast_div(f, s.by_chunks), c = f - block * s.chunks;
      const int nt = min((n_base >> 5) + block, last_nt);  // blocks past N: any weights, their results are not stored
      const uint8_t* src = bp + (static_cast<int64_t>(nt) * s.packed_kt + c) * kChunkBytes + ((lane & 32) + ch) * 16;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                       (__attribute__((address_space(3))) void*)(lds + f * kChunkBytes), 16, 0, 0);
    }
  }
  for (int i = threadIdx.x; i < channels; i += 256) {
    int comp;
    float scale, bias;
    resolve_channel(e, min(n_base + i, s.N - 1), s.N, &comp, &scale, &bias);
    p_comp[i] = comp;
    p_scale[i] = scale;
    p_bias[i] = bias;
  }
  if constexpr (CONV && !HOLD) {
    for (int p = threadIdx.x; p < (s.K >> 4); p += 256) table[p] = window_piece(p);
  }
  wait_vmcnt<0>();  // the direct loads of this wavefront have landed
  __syncthreads();

  if (n0 >= s.N || t0 >= t1) return;  // whole wavefront; no barrier follows
  const int chunks = HOLD ? GROUP : s.chunks;
  const uint8_t* const wfrag = lds + wn * kBlocks * s.chunks * kChunkBytes + lane * 16;
  const int groups = (s.chunks + GROUP - 1) / GROUP;
  // Rows that a wavefront writes whole are contiguous in memory and go out as streaming stores, ahead of the flush of L2 at
  // the end of the kernel (401408 x 32 -> 64: 12.2 -> 10.9 us); of longer rows it writes 64 bytes here and there, which L2
  // has to put together first (100352 x 64 -> 256 with the residual: 18.8 us streaming, 15.5 us plain).
  const bool stream_out = s.N <= kBlocks * 32;
  for (int tile = t0; tile < t1; ++tile) {
    if (tile + 1 < t1) load_add(tile + 1, add_nxt);  // a whole tile ahead: these come from memory
    // the lane's channels in the parameter panels, hidden from the compiler: it would keep all 96 parameters of a lane in
    // registers across the loop and spill
    int col0 = wn * kBlocks * 32 + half * 16;
    asm volatile("" : "+v"(col0));
    v16i acc[kBlocks];
#pragma unroll
    for (int b = 0; b < kBlocks; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v4i c = *reinterpret_cast<const v4i*>(p_comp + col0 + b * 32 + g * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[b][g * 4 + r] = c[r];
      }
    auto weight = [&](int c, v4i (&w)[kBlocks]) {
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) w[b] = *reinterpret_cast<const v4i*>(wfrag + (b * chunks + c) * kChunkBytes);
    };
    auto multiply = [&](v4i x, const v4i (&w)[kBlocks]) {
      x.x ^= amask; x.y ^= amask; x.z ^= amask; x.w ^= amask;
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) acc[b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[b], x, acc[b], 0, 0, 0);
    };
    if constexpr (HOLD) {
      // The weight comes from LDS a chunk ahead (with each chunk waiting for its own reads 13.0 us instead of 12.8).  The
      // branch on `more` stays between the chunks: without it the scheduler reads all of them first and spills.
      const bool more = tile + 1 < t1;  // wavefront uniform
      if (more) locate(tile + 1);
      v4i w[2][kBlocks];
      weight(0, w[0]);
#pragma unroll
      for (int u = 0; u < GROUP; ++u) {
        if (u + 1 < GROUP) weight(u + 1, w[(u + 1) & 1]);
        multiply(cur[u], w[u & 1]);
        if (more) cur[u] = load_held(u);
      }
    } else {
      for (int g = 0; g < groups; ++g) {
        // the next group (of this tile, or the first of the next one) travels under this group's MFMAs
        if (g + 1 < groups) {
#pragma unroll
          for (int u = 0; u < GROUP; ++u) nxt[u] = load(min((g + 1) * GROUP + u, s.chunks - 1));
        } else if (tile + 1 < t1) {
          locate(tile + 1);
#pragma unroll
          for (int u = 0; u < GROUP; ++u) nxt[u] = load(min(u, s.chunks - 1));
        }
#pragma unroll
        for (int u = 0; u < GROUP; ++u) {
          const int c = g * GROUP + u;
          if (c < s.chunks) {  // wavefront uniform
            v4i w[kBlocks];
            weight(c, w);
            multiply(cur[u], w);
          }
        }
#pragma unroll
        for (int u = 0; u < GROUP; ++u) cur[u] = nxt[u];
      }
    }
    v4i packed[kBlocks];
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int col = col0 + b * 32 + g * 4;
        const f4 sc = *reinterpret_cast<const f4*>(p_scale + col);
        const f4 bi = *reinterpret_cast<const f4*>(p_bias + col);
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = static_cast<float>(acc[b][g * 4 + r]) * sc[r];
          v[r] = v[r] + bi[r];
          if constexpr (SUM == 1) v[r] = v[r] + s.sum_scale * static_cast<float>((static_cast<uint32_t>(add[b][g]) >> (8 * r)) & 0xffu);
          if constexpr (SUM == 2) v[r] = v[r] + s.sum_scale * static_cast<float>((add[b][g] << (24 - 8 * r)) >> 24);
          if constexpr (POST == kPostRelu && OUT_T != ITEXHIP_QUINT8) v[r] = fmaxf(v[r], 0.0f);
          if constexpr (POST == kPostClip) v[r] = __builtin_amdgcn_fmed3f(v[r], s.lo, s.hi);  // lo <= hi; lo for NaN, as min(max()) gives
        }
        packed[b][g] = static_cast<int>(pack_bytes<OUT_T, POST>(v));
      }
    }
    // A lane holds pieces (16 channels) `half` and 2 + half of its row.  Rows 16 .. 31 of the first trade places with rows
    // 0 .. 15 of the second: then a store covers the 64 bytes of 16 rows instead of 32 bytes of 32 rows.
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const auto t = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(packed[0][g]), static_cast<uint32_t>(packed[1][g]), false, false);
      packed[0][g] = static_cast<int>(t[0]);
      packed[1][g] = static_cast<int>(t[1]);
    }
    const int n = n0 + (half + 2 * (lrow >> 4)) * 16;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int m = tile * 32 + b * 16 + (lrow & 15);
      v4i* const dst = reinterpret_cast<v4i*>(out + (static_cast<uint32_t>(m) * static_cast<uint32_t>(s.N) + static_cast<uint32_t>(n)));
      if (m < s.M && n < s.N) {
        if (stream_out) __builtin_nontemporal_store(packed[b], dst);
        else *dst = packed[b];
      }
    }
    if constexpr (SUM != 0) {
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) add[b] = add_nxt[b];
    }
  }
}

template <int OUT_T, int POST, int SUM, int GROUP, bool CONV, bool HOLD>
int launch(const uint8_t* a, uint32_t amask, const uint8_t* bp, const StreamArgs& s, const EpilogueArgs& e, uint8_t* out,
           const ConvTileArgs& cv, dim3 grid, size_t lds, hipStream_t st) {
  auto kern = qgemm_stream_kernel<OUT_T, POST, SUM, GROUP, CONV, HOLD>;
  static unsigned long long attr_done = 0;  // devices on which this instantiation's attribute is set
  if (!device_bit(&attr_done, false)) {
    hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (err != hipSuccess) return hip_fail(err, "hipFuncSetAttribute(qgemm_stream_kernel)");
    device_bit(&attr_done, true);
  }
  note_kernel(kLastShortK, GROUP * 100 + HOLD);
  kern<<<grid, 256, lds, st>>>(a, amask, bp, s, e, out, cv);
  return ITEXHIP_OK;
}

template <int OUT_T, int GROUP, bool CONV, bool HOLD, bool SUMS>  // SUMS: with a residual
int dispatch(const uint8_t* a, uint32_t amask, const uint8_t* bp, const StreamArgs& s, int post, const EpilogueArgs& e, uint8_t* out,
             const ConvTileArgs& cv, dim3 grid, size_t lds, hipStream_t st) {
#define STREAM(P, S) return launch<OUT_T, P, S, GROUP, CONV, HOLD>(a, amask, bp, s, e, out, cv, grid, lds, st)
  if constexpr (SUMS) {
    const bool u8 = e.addend_type == ITEXHIP_QUINT8;
    switch (post) {
      case kPostNone: if (u8) STREAM(kPostNone, 1); else STREAM(kPostNone, 2);
      case kPostRelu: if (u8) STREAM(kPostRelu, 1); else STREAM(kPostRelu, 2);
      default: if (u8) STREAM(kPostClip, 1); else STREAM(kPostClip, 2);
    }
  } else {
    switch (post) {
      case kPostNone: STREAM(kPostNone, 0);
      case kPostRelu: STREAM(kPostRelu, 0);
      default: STREAM(kPostClip, 0);
    }
  }
#undef STREAM
}

}  // namespace

// 1: the call was launched here; 0: not a call for this kernel; < 0: an error (the status, negated).
int try_stream(const uint8_t* a, uint32_t amask, const uint8_t* bp, int M, int K, int N, const EpilogueArgs& e, int out_type,
               void* out, hipStream_t st, const ConvTileArgs* cv) {
  if (out_type != ITEXHIP_QUINT8 && out_type != ITEXHIP_QINT8) return 0;
  const int forced = __atomic_load_n(&g_forced_tile_shape[cv ? 1 : 0], __ATOMIC_RELAXED);  // tests ask for a tile shape, or
  if (forced >= 0 && forced != kForceStream) return 0;                                     // for this kernel at any size
  if (K % 16 != 0 || K < 16 || N % 16 != 0 || (e.bias == nullptr && !e.fused) || !aligned(out, 16) || e.row_min_a) return 0;
  if (static_cast<int64_t>(M) * N >= (1LL << 31)) return 0;
  CanonChain c;
  const int act = canon_chain(e, &c);
  if ((c.flags & kChainClip) && !(c.lo <= c.hi)) return 0;  // the median of three is no clip then
  if (act < 0 || act > 2 || (c.flags & ~(kChainMax0 | kChainClip | kChainSumFirst)) != 0) return 0;
  if (e.addend && (!(c.flags & kChainSumFirst) || (e.addend_type != ITEXHIP_QUINT8 && e.addend_type != ITEXHIP_QINT8) ||
                   !aligned(e.addend, 4)))
    return 0;
  StreamArgs s{};
  s.M = M; s.K = K; s.N = N;
  s.chunks = (K + 31) / 32;
  s.by_chunks = make_fast_div(s.chunks);
  s.packed_kt = 2 * ((K + 63) / 64);
  const int cols = (N + kBlocks * 32 - 1) / (kBlocks * 32);  // wavefront columns
  s.waves_n = cols >= 4 ? 4 : cols >= 2 ? 2 : 1;
  while (s.waves_n > 1 && s.waves_n * kBlocks * s.chunks * kChunkBytes > kMaxWeightBytes) s.waves_n >>= 1;
  const int weight = s.waves_n * kBlocks * s.chunks * kChunkBytes;
  if (weight > kMaxWeightBytes) return 0;
  s.tiles = (M + 31) / 32;
  // Where it is the faster kernel, by what fills the device: `rounds` is how often the 32 x 64 pieces of the result go into
  // the 4096 wavefronts that run at once (in quarters).  Below one round a launch is its start, and without a residual the tile kernel starts
  // sooner; with a long K the MFMAs and the weight fragments read from LDS for every 32 rows count, and the tile kernel
  // reads them for 64 - 256; past K = 384 the weight of 128 channels leaves room for two workgroups per CU instead of three or
  // four.  Tile kernel / this kernel, time, over 16 to 14336 channels (convolutions: 32 to 512), at about 0.8, 1, 1.5, 2 and 4
  // rounds (the tile kernel's own steps, whole tiles per CU, are in it):
  //   K <= 48                 1.0 - 1.4, 1.0 - 1.5, 1.1 - 1.7, 1.3 - 1.9, 1.5 - 2.1   with a residual 1.2 - 2.2 everywhere
  //   K = 64                  1.0 - 1.4, 0.9 - 1.3, 1.0 - 1.4, 1.0 - 1.6, 1.1 - 2.0   with a residual 1.0 - 2.9
  //                           (up to 1.0 before 1.75 rounds: multiples of 128 channels from 256 on)
  //   K = 80, 96, 112         0.9 - 1.4, 0.9 - 1.4, 1.0 - 1.5, 1.1 - 1.7, 1.3 - 2.1   with a residual 0.9 - 1.8, 1.0 - 2.0
  //   K = 128                 0.8 - 1.2, 0.8 - 1.1, 0.7 - 1.2, 0.8 - 1.3, 1.0 - 1.7   with a residual 0.9 - 1.8, 0.8 - 1.6, 0.8 -
  //                           1.5, 0.9 - 2.0, 1.0 - 2.5 (below 1: multiples of 128 channels, 1 to 2 rounds, over 1024 to 2.75)
  //   K = 144, 160            0.8 - 1.3, 0.9 - 1.3, 1.0 - 1.4, 1.0 - 1.6, 1.2 - 1.9   with a residual 0.9 - 2.1, from 1.25 on 1.1
  //   longer, up to 1024 channels (2048 with a residual)
  //     K = 192, 256, 320, 448  0.7 - 1.2, 0.7 - 1.1, 0.7 - 1.3, 0.8 - 1.3, 1.0 - 1.7   with a residual 1.0 - 2.9 at 4
  //     K = 208 ... 480, no 64 n  0.7 - 1.3, 0.8 - 1.4, 0.9 - 1.5, 1.0 - 1.6, 1.1 - 1.9   with a residual 1.0 - 2.0 from 1.5 on
  //     K = 512                 0.7 - 0.9, 0.7 - 1.1, 0.7 - 1.1, 0.7 - 1.0, 0.9 - 1.1 (also at 6 and 8), 128 channels 1.1 - 1.2;
  //                             with a residual 1.3 - 1.6 at 4
  //   longer, more channels (few rows per wavefront, workgroups that do not fill the last pass): 1.5 rounds, 2, 4, 6 and more
  //     K = 192, 256            0.7 - 0.9, 0.7 - 0.9, 0.8 - 0.9, 0.7 - 1.0   with a residual (192) 1.1 at 4, 1.2 - 1.3; (256) 0.7 - 1.0
  //     K = 208                 1.0, 1.05, 1.15, 1.0 - 1.3                   with a residual 1.0 - 1.1, 1.0 - 1.2, 1.3, 1.2 - 1.5
  //     K = 272 ... 480         0.7 - 1.0, 0.8 - 1.0, 0.9 - 1.0, 0.7 - 1.1   with a residual 0.9 - 1.2, 0.9 - 1.3, 1.1 - 1.6, 1.0 - 1.7
  //   up to 256 deep all K chunks of a tile are held at once; without a residual, 0.75, 1, 1.5, 2.5 and 3.5 rounds (the ranges above were
  //   measured over more channels, and before the chunks were held):
  //     up to 64 channels     K = 128 1.0, 1.1 - 1.2, 1.3, 1.4, 1.4;  144, 160 1.2 - 1.3, 1.2, 1.35 - 1.45, 1.4 - 1.5, 1.5;  176 to 256
  //                           1.05 - 1.15, 1.15 - 1.25, 1.25 - 1.35, 1.3 - 1.5, 1.3 - 1.5 (100352 x 256 -> 64 9.5 -> 8.1 us;
  //                           only with both tensors in L2, launch after launch, one column is 0.9 - 1.2: 6.8 -> 7.9)
  //     65 to 1024            K = 128 -, -, 0.85 - 1.0, 0.9 - 1.1 (96 and 192 channels 1.3 - 1.7), 1.07 - 1.8, at 3 rounds 1.05 - 1.6;
  //                           K = 192 -, 0.8, 1.0 - 1.5 (768 at 1.75 0.9), 1.1 - 1.8, 1.3 - 1.9, at 2 rounds 1.1 - 1.5;  K = 256 0.9 up to 2, 1.0 at 3
  //   with a residual, small launches: 16 to 4096 channels at 0.15, 0.25, 0.5, 0.75, 1 and 1.25 rounds (a MatMul; 128 x 128 tiles start late there)
  //     K <= 64               1.0 - 1.1, 1.0 - 1.6, 1.2 - 2.2, 1.2 - 2.0;  80 to 112  0.9 - 1.1, 1.0 - 1.6, 1.0 - 1.4, 1.1 - 1.5
  //     K = 128               0.9 - 1.1, 0.9 - 1.1, 1.1 - 1.9, 1.1 - 1.7, 1.0 - 1.3, 1.05 - 1.3 (from 1024 channels on 0.9 - 1.0), then 1.0 - 2.5
  //     K = 160               0.9 - 1.0, 1.0 - 1.4, 1.0 - 1.4, 1.05 - 1.4, 1.0 - 1.5, 1.0 - 1.5
  //     K = 192; 256          0.8 - 1.0, 0.9 - 1.1, 1.2 - 1.9, 1.1 - 1.7, 1.0 - 1.2, 1.0 - 1.2;  0.8 - 0.9, 0.8 - 0.95, 1.0 - 1.7, 1.05 - 1.5, 0.9 - 1.1, 0.9 - 1.1
  //   convolution, K <= 384   1.0 - 1.3, 1.0 - 1.2, 1.2 - 1.5, 1.1 - 1.5, 1.7         with a residual 1.1 - 1.7
  //                           over 256 channels and K 192 to 288: 0.8 - 1.2, 0.9 - 1.2, 1.0 - 1.4, 1.0 - 1.6, 1.1 - 2.0, but K = 288
  //                           with three columns of workgroups (over 256 to 384 channels, the activations gathered three
  //                           times) 0.7 - 0.9, 0.7 - 0.9, 0.7 - 1.1, 0.7 - 1.1, 0.75 - 1.1, from 6 on 1.05 - 1.2
  //   convolution, K <= 448   up to 64 channels 1.1, 1.05, 1.15, -, -; more 1.0, 0.9, 1.1, 0.9, 0.9   with a residual
  //                           1.1 - 1.2, 0.95 - 1.0, 1.3, 0.9 - 1.0, 0.9 - 1.05
  //   convolution, K = 576    0.9 - 1.1, 1.0, 1.15, -, -                              K = 1152: 0.87 - 0.94
  const int64_t quarter_rounds = static_cast<int64_t>(s.tiles) * cols / 1024;
  auto within = [&](int64_t least, int64_t most = INT64_MAX) { return quarter_rounds >= least && quarter_rounds <= most; };
  const bool sum = e.addend != nullptr, wide = N > 64, very_wide = N > (sum ? 2048 : 1024);
  const bool whole = K % 64 == 0, fits = whole && N % 128 == 0;  // nothing padded in the tile kernel
  bool take;
  if (cv) {
    take = conv_streams(K, N, sum, quarter_rounds);
  } else if (K <= 64) {
    take = within(sum ? 1 : fits && N >= 256 ? 7 : 4);
  } else if (K < 128) {
    take = within(sum ? 1 : 6);
  } else if (K == 128) {
    take = sum ? within(2) && !(fits && N >= 1024 && within(4, 5)) : within(!wide ? 4 : very_wide ? 16 : 12);
  } else if (K <= 160) {
    take = within(sum ? 2 : !wide ? 3 : 6);
  } else if (K <= 256 && !wide && !sum) {
    take = within(3);
  } else if (K == 192 && !very_wide && !sum) {
    take = within(8);
  } else if (K <= 512) {
    take = within(whole ? 16 : very_wide ? (sum && K <= 352 ? 12 : 16) : K <= 288 && !sum && N % 128 == 0 ? 7 : 6);
    if (very_wide) take = take && (sum ? K != 256 : K <= 224 && !whole);
    if (sum && (K == 192 ? within(2, 5) : K == 256 && within(2, 3))) take = true;
    if (K == 512) take = take && (sum || N == 128);
    else if (K > 448 && !wide) take = take && within(6, 12);
  } else {
    take = false;
  }
  if (forced != kForceStream && !take) return 0;
  s.padded = cv && (cv->pad_top > 0 || cv->pad_left > 0 ||
                    (cv->out_h - 1) * cv->stride_h + (K / (cv->k_w * cv->in_c) - 1) * cv->dil_h >= cv->in_h ||
                    (cv->out_w - 1) * cv->stride_w + (cv->k_w - 1) * cv->dil_w >= cv->in_w);
  // (Input and result past 384 MB: not held where three columns of wavefronts leave every fourth one idle, 0.67 - 1.02 of the time
  // held (0.80 in the middle), nor with up to 4 chunks over more than 768 channels, 0.75 - 1.04 (0.86); below, and elsewhere,
  // held chunks are 1.1 times as fast in the mean.  700 sizes.)
  const int64_t conv_bytes = cv ? static_cast<int64_t>(M) * N + static_cast<int64_t>(M / cv->out_w / cv->out_h) * cv->in_h * cv->in_w * cv->in_c : 0;
  const bool conv_early = conv_bytes > (384 << 20) && (cols == 3 || (s.chunks <= 4 && cols > 12));
  const bool held_conv = cv && !sum && !s.padded && s.chunks <= 8 && !conv_early;
  const size_t lds = static_cast<size_t>(weight) + 12 * s.waves_n * kBlocks * 32 + (cv && !held_conv ? (K >> 4) * 8 : 0);
  const int per_cu = std::min<int>(4, 160 * 1024 / static_cast<int>(lds));  // 128 registers: four wavefronts per SIMD
  const int groups_n = (cols + s.waves_n - 1) / s.waves_n;
  if (groups_n > 65535) return 0;  // gridDim.y
  const int waves_m = 4 / s.waves_n;
  // as many workgroups on every XCD (the kernel gives each a contiguous range of them): 2048 x 400 -> 6144, 10 of 16 with work
  // and all of it on five XCDs, 24.8 us
  s.walkers = std::min(s.tiles, 8 * std::max(1, 32 * per_cu / groups_n) * waves_m);
  s.share = (static_cast<uint64_t>(s.tiles) << 24) / s.walkers;
  const int wgs = (s.walkers + waves_m - 1) / waves_m;
  const dim3 grid(static_cast<unsigned>((wgs + 7) / 8 * 8), static_cast<unsigned>(groups_n));
  s.lo = c.lo; s.hi = c.hi; s.sum_scale = c.sum_scale;
  const int post = c.flags & kChainClip ? kPostClip : c.flags & kChainMax0 ? kPostRelu : kPostNone;
  uint8_t* o = static_cast<uint8_t*>(out);
  int rc;
  const bool u8 = out_type == ITEXHIP_QUINT8;
#define STREAM(G, CONV, HOLD, SUMS, GEO)                                                                                  \
  rc = u8 ? dispatch<ITEXHIP_QUINT8, G, CONV, HOLD, SUMS>(a, amask, bp, s, post, e, o, GEO, grid, lds, st)                \
          : dispatch<ITEXHIP_QINT8, G, CONV, HOLD, SUMS>(a, amask, bp, s, post, e, o, GEO, grid, lds, st)
  const ConvTileArgs none{};
#define HELD(CONV, SUMS, GEO)                                  \
  case 1: STREAM(1, CONV, true, SUMS, GEO); break;             \
  case 2: STREAM(2, CONV, true, SUMS, GEO); break;             \
  case 3: STREAM(3, CONV, true, SUMS, GEO); break;             \
  case 4: STREAM(4, CONV, true, SUMS, GEO); break
#define HELD_LONG(CONV, GEO)                                   \
  case 5: STREAM(5, CONV, true, false, GEO); break;            \
  case 6: STREAM(6, CONV, true, false, GEO); break;            \
  case 7: STREAM(7, CONV, true, false, GEO); break;            \
  case 8: STREAM(8, CONV, true, false, GEO); break
  if (cv && sum) {
    STREAM(2, true, false, true, *cv);
  } else if (cv) {
    switch (held_conv ? s.chunks : 0) {
      HELD(true, false, *cv);
      HELD_LONG(true, *cv);
      default: STREAM(4, true, false, false, *cv);
    }
  } else if (sum) {
    // Held, or groups of 1, 2 or 4 (4 with a residual spills up to 4 registers, which a long K covers).  Held chunks need the
    // caches: past 256 MB of activations, residual and result, or past 96 MB where rows are no multiple of 64 bytes and pieces
    // of lines have to meet in them, the groups' earlier loads win.  Time over that of groups of 1 (one chunk), 2 (two) or 4
    // (more), 3000 sizes:
    //   chunks 1 - 4   held: below the lines 0.8 - 1.1, between them with ragged rows 0.86 - 1.25 (1.02 in the middle), past
    //                  both 1.05 - 1.39 (323916 x 112 -> 528 118 -> 169 us); groups of 2 there 0.82 - 1.08
    //   chunks 5 - 9   groups of 2 0.82 - 1.09 (0.97 in the middle), past 256 MB 1.0 - 1.1
    //   chunks 10 - 12 groups of 2 0.84 - 1.07 everywhere;  13 - 16  0.98 - 1.25 (368813 x 464 -> 176 113 -> 142 us)
    const int64_t bytes = static_cast<int64_t>(M) * K + 2 * static_cast<int64_t>(M) * N;
    const bool cached = bytes <= ((N % 64 == 0 || s.chunks > 4 ? 256 : 96) << 20);
    if (s.chunks > 12 || (s.chunks > 4 && s.chunks <= 9 && !cached)) {
      STREAM(4, false, false, true, none);
    } else if (s.chunks == 1 && !cached) {
      STREAM(1, false, false, true, none);
    } else {
      switch (cached ? s.chunks : 0) {
        HELD(false, true, none);
        default: STREAM(2, false, false, true, none);
      }
    }
  } else {
    // Held chunks need the caches here too: past `line` MB of activations and result the groups' earlier loads win, but not for
    // one column of wavefronts, nor everywhere for a longer K.  Groups of 1, 2 or 4 over held chunks, time, 2800 sizes (the
    // middle in brackets):
    //   chunks 1 - 4   past 384 MB over 65 to 128 channels 0.74 - 1.01 (0.88), over 193 and more 0.68 - 1.16 (0.82: 94214 x 48 -> 7024
    //                  275 -> 191 us); over 129 to 192, two workgroups abreast and a column of the second idle, 1.0 - 1.27 (1.17) up
    //                  to 448 MB, 0.67 - 1.15 (0.94) past them; over more than 448 channels one chunk from 320 MB on 0.85 - 1.05
    //                  (0.96), two chunks from 128 to 180 MB 0.82 - 0.95 (0.93) and up to 384 MB 0.75 - 1.1 (0.99)
    //                  else, up to the lines, 0.81 - 1.4 (1.02)
    //   chunks 5 - 8   up to 384 MB 0.69 - 1.40 (1.12);  past them over 65 to 192 channels 0.61 - 0.96 (0.89), more 0.79 - 1.53
    //                  (1.05: not there)
    const int64_t bytes = static_cast<int64_t>(M) * (K + N);
    const int64_t line = s.chunks > 4 ? 384 : cols == 3 ? 448 : cols >= 8 && s.chunks == 1 ? 320 : cols >= 8 && s.chunks == 2 ? 128 : 384;
    const bool early = bytes > (line << 20) && cols >= 2 && (s.chunks <= 4 || cols <= 3);
    if (early && s.chunks == 1) {
      STREAM(1, false, false, false, none);
    } else if (early && s.chunks == 2) {
      STREAM(2, false, false, false, none);
    } else {
      switch (early ? 0 : s.chunks) {
        HELD(false, false, none);
        HELD_LONG(false, none);
        default: STREAM(4, false, false, false, none);
      }
    }
  }
#undef HELD_LONG
#undef HELD
#undef STREAM
  return rc == ITEXHIP_OK ? 1 : -rc;
}

}  // namespace itexhip
