// Quantized BatchMatMul by bands of 16 output rows (itex/core/kernels/common/batch_matmul_op.h:36-522): the calls of qbmm.hip whose
// x is not transposed and whose fused operands do not depend on the row, where the rule at the end of this file says so.
//
// A workgroup stages y in LDS once, k-contiguous per output column, and each of its four wavefronts computes bands of 16 rows by
// itself: x from memory to v_mfma_i32_16x16x64_i8 (y as the first operand: a lane gets four neighbouring columns of one row), the
// results by 8- and 16-byte writes into an image of the band in LDS, and the image, which is contiguous in the output, out in
// aligned 16-byte streaming stores, whole lines whatever the row length; no barrier after the first.  Rows that are no
// whole 16-byte vectors stand in the image at a pitch of their own, and the first elements of a row once more behind the row above
// it, so that a vector of the output is always contiguous there; it is fetched by three aligned 8-byte reads and shifted (an
// unaligned LDS read takes a cycle per lane, 64 for what 4 do; an unaligned write 8 for 2).
//
// Bound by vector instructions (some 22 per 16 x 16 tile of Q.K^T with two operands, 18 of them the conversion, the three
// roundings and the narrowing) and the start of the launch.  us, 64 x 64 and 128 x 128 tiles -> bands, one MI355X: 384 products of
// 197 x 64 by 64 x 197 with Mul + Add, bfloat16 16.4 -> 12.3, fp32 41.0 -> 20.8; 197 x 197 by 197 x 64 to bfloat16 10.8 -> 8.8.  Also
// measured: the four wavefronts sharing each band's columns (a quarter of the image, two barriers per band): 12.3 -> 16.0 and
// 8.8 -> 22, better only for fp32 rows of 383 columns (31 -> 22).
#include <algorithm>

#include "qbmm_stage.hpp"

namespace itexhip {
namespace {

constexpr int kBand = 16;      // output rows of a band
constexpr int kBandWaves = 4;
constexpr int kMaxKTiles = 6;

struct BandArgs {
  itexhip_bmm_params p;
  FastDiv by_dim[ITEXHIP_BMM_MAX_BATCH_DIMS];
  FastDiv by_row;               // elements of an output row, or (rows of whole vectors) its 16-byte vectors
  uint32_t batch;
  int xcd_grid;                 // launched as (8, parts, matrices / 8), not (parts, matrices)
  int bands, bands_per_part;
  int rows16, k_tiles;          // columns of the output in LDS, a multiple of 16; k tiles of 64
  int whole_rows;               // output rows are whole aligned 16-byte vectors
  int chunk, chunks;            // columns of the output that a workgroup computes: all, or (whole rows) a part of them
  int pitch, band_bytes;        // of a band's image in LDS
  int operand_at[ITEXHIP_BMM_MAX_BINARY], bands_at;  // LDS offsets
  int step_rows, step_cols;     // 64 vectors on in the output: so many rows and elements
};

typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u2_any __attribute__((ext_vector_type(2), aligned(2)));

// 16 bytes at base + at (wave-uniform base).  Written through for the product that the attention block reads again (streaming stores
// are faster by themselves, and what reads the result waits longer: 128 x 128 tokens, P.V to bfloat16 + QuantizeV2 8.7 + 5.0 us
// streaming, 8.6 + 4.3 written through, 9.6 + 4.3 plain) and for 16-bit results; fp32 scores stream.
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
template <bool STREAM>
__device__ __forceinline__ void store16(char* base, int at, v4i v) {
  constexpr int kCacheStream = 2, kCacheThrough = 17;  // nt; sc0 sc1
  const auto r = __builtin_amdgcn_make_buffer_rsrc(base, 0, 0x7fffffff, 0x00027000);
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, at, 0, STREAM ? kCacheStream : kCacheThrough);
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// y in LDS: per k tile of 64 the output columns' bytes, 64 each, their 16-byte pieces rotated (piece p of column n in place
// p ^ (n / 4) % 4: the fragment reads of 16 columns meet no bank twice).  Where y is transposed on the way 64 bytes of space stand
// behind every 16 columns, so that its writes do not either.
constexpr int tile16_bytes(bool adj_y) { return 16 * kTile + (adj_y ? 0 : 64); }
template <bool ADJ_Y>
__device__ __forceinline__ int y_piece(int n, int piece) {
  return (n >> 4) * tile16_bytes(ADJ_Y) + (n & 15) * kTile + (piece ^ ((n >> 2) & 3)) * 16;
}

template <bool ADJ_Y, int MODE, int NB, int OUT_T, int KT>
__global__ __launch_bounds__(64 * kBandWaves, 4) void qbmm_band_kernel(const BandArgs a, const int8_t* __restrict__ x_all,
                                                                       const int8_t* __restrict__ y_all, char* __restrict__ out) {
  using elem_t = typename std::conditional<OUT_T == ITEXHIP_FLOAT, float, uint16_t>::type;
  constexpr int ESZ = sizeof(elem_t), VE = 16 / ESZ, TILE16 = tile16_bytes(ADJ_Y);
  constexpr bool STREAM = OUT_T == ITEXHIP_FLOAT && ADJ_Y;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const itexhip_bmm_params& p = a.p;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t bi = a.xcd_grid ? blockIdx.z * 8 + blockIdx.x : blockIdx.y;
  const int job = a.xcd_grid ? blockIdx.y : blockIdx.x;
  if (bi >= a.batch) return;
  const int M = static_cast<int>(p.M), K = static_cast<int>(p.K), N = static_cast<int>(p.N);
  const int part = a.chunks == 1 ? job : job / a.chunks, n_first = a.chunks == 1 ? 0 : (job - part * a.chunks) * a.chunk;

  // (every dimension, the missing ones of extent 1: straight-line code whose arguments arrive together)
  int64_t xo = 0, yo = 0, bo[ITEXHIP_BMM_MAX_BINARY] = {0, 0};
  uint32_t rem = bi;
#pragma unroll
  for (int d = ITEXHIP_BMM_MAX_BATCH_DIMS - 1; d >= 0; --d) {
    const uint32_t q = d == 0 ? 0 : static_cast<uint32_t>(fast_div(static_cast<int>(rem), a.by_dim[d]));
    const uint32_t i = rem - q * static_cast<uint32_t>(p.batch_dims[d]);
    rem = q;
    xo += i * p.x_batch_stride[d];
    yo += i * p.y_batch_stride[d];
#pragma unroll
    for (int b = 0; b < NB; ++b) bo[b] += i * p.binary[b].batch_stride[d];
  }
  const int8_t* x = x_all + xo;
  const int8_t* y = y_all + yo;

  // A band's x: lane l multiplies 16 k of row l % 16.  kAligned: it loads them.  kAny: lane l loads 16 k of row l / 4, four lanes
  // a row's 64 bytes, and the piece moves through LDS (unaligned loads whose neighbouring lanes lie in different rows take long:
  // P.V over 383 tokens 13.2 -> 9.5 us; where loads are aligned the way through LDS costs as much as it gives).
  const int last = M * K - 16, x_row = MODE == kAligned ? lane & 15 : lane >> 2, x_k = (MODE == kAligned ? lane >> 4 : lane & 3) * 16;
  v4i xf[KT];
  auto load_x = [&](int m0) {
    const int row = min(m0 + x_row, M - 1) * K;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      if (KT > 1 && kt >= a.k_tiles) break;
      const int k = kt * kTile + x_k;
      if constexpr (MODE == kAligned) xf[kt] = *reinterpret_cast<const v4i*>(x + (k < K ? row + k : 0));
      else xf[kt] = *reinterpret_cast<const v4i_any*>(x + min(row + k, last));
    }
  };
  auto turn_x = [&](int m0, uint8_t* scratch) {
    if constexpr (MODE == kAligned) return;
    const int row = min(m0 + x_row, M - 1) * K + x_k;
    const bool settle = (min(m0 + kBand, M) - 1) * K + a.k_tiles * kTile > M * K;  // the same for the wavefront
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      if (KT > 1 && kt >= a.k_tiles) break;
      if (settle) xf[kt] = shift_down(xf[kt], static_cast<uint32_t>(max(row + kt * kTile - last, 0)) & 15u);
      *reinterpret_cast<v4i*>(scratch + kt * 1024 + y_piece<ADJ_Y>(lane >> 2, lane & 3)) = xf[kt];
    }
    wave_sync();
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      if (KT > 1 && kt >= a.k_tiles) break;
      xf[kt] = *reinterpret_cast<const v4i*>(scratch + kt * 1024 + y_piece<ADJ_Y>(lane & 15, lane >> 4));
    }
    wave_sync();
  };

  const int band_end = min((part + 1) * a.bands_per_part, a.bands);
  int band = part * a.bands_per_part + wave;
  if (band < band_end) load_x(band * kBand);

  float uniform[NB > 0 ? NB : 1];
  const int k_bytes = a.rows16 / 16 * TILE16;  // of a k tile
  // the fused operands, widened, n contiguous: requested ahead of y, put into LDS behind it
  elem_t first[NB > 0 ? NB : 1];
  auto operand = [&](int b, int n) {
    return (static_cast<const elem_t*>(p.binary[b].data) + bo[b])[min(n_first + n, N - 1) * p.binary[b].stride_n];
  };
#pragma unroll
  for (int b = 0; b < NB; ++b) first[b] = operand(b, t);
  if constexpr (ADJ_Y) {  // a thread: 16 k of a column, aligned; k fastest over the threads
    static_assert(MODE == kAligned, "the rule takes no unaligned operands where y lies along k");
    const int units = a.rows16 * a.k_tiles * 4;
    for (int u0 = t; u0 < units; u0 += 4 * 64 * kBandWaves) {
      v4i w[4];
      int n[4], k[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = min(u0 + u * (64 * kBandWaves), units - 1) >> 2;
        const int kt = KT == 1 ? 0 : i / a.rows16;
        n[u] = i - kt * a.rows16;
        k[u] = kt * kTile + (t & 3) * 16;
        w[u] = *reinterpret_cast<const v4i*>(y + (k[u] < K ? min(n_first + n[u], N - 1) * K + k[u] : 0));
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (k[u] >= K) w[u] = v4i{0, 0, 0, 0};  // (K is a multiple of 16)
        if (u0 + u * (64 * kBandWaves) < units) *reinterpret_cast<v4i*>(lds + (k[u] >> 6) * k_bytes + y_piece<ADJ_Y>(n[u], t & 3)) = w[u];
      }
    }
  } else {  // a thread: 4 k of 16 columns, transposed four columns at a time; columns fastest over the threads
    const int groups = a.rows16 >> 4, units = groups * a.k_tiles * 16;
    for (int u = t; u < units; u += 64 * kBandWaves) {
      const int kq = u / groups, n = (u - kq * groups) * 16, col = n_first + n;
      v4i w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int8_t* row = y + min(kq * 4 + i, K - 1) * N;
        w[i] = *reinterpret_cast<const v4i_any*>(row + min(col, N - 16));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (col > N - 16) w[i] = shift_down(w[i], static_cast<uint32_t>(col - (N - 16)) & 15u);
        if (kq * 4 + i >= K) w[i] = v4i{0, 0, 0, 0};
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t rows[4] = {static_cast<uint32_t>(w[0][j]), static_cast<uint32_t>(w[1][j]), static_cast<uint32_t>(w[2][j]),
                                  static_cast<uint32_t>(w[3][j])};
        uint32_t v[4];
        transpose_4x4(rows, v);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<uint32_t*>(lds + (kq >> 4) * k_bytes + y_piece<ADJ_Y>(n + j * 4 + i, (kq >> 2) & 3) + (kq & 3) * 4) = v[i];
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    uniform[b] = widen<OUT_T>(first[b]);
    if (p.binary[b].stride_n == 0) continue;
    for (int n = t; n < a.rows16; n += 64 * kBandWaves) reinterpret_cast<float*>(lds + a.operand_at[b])[n] = widen<OUT_T>(n == t ? first[b] : operand(b, n));
  }
  __syncthreads();

  uint8_t* image = lds + a.bands_at + wave * a.band_bytes;
  uint8_t* mine = image + (lane & 15) * a.pitch + (lane >> 4) * (4 * ESZ);
  const uint8_t* frag = lds + (lane & 15) * kTile + ((lane >> 4) ^ ((lane >> 2) & 3)) * 16;
  const float scale = p.scale;
  const int tiles16 = a.rows16 >> 4;
  // G column tiles from tile `base` on: product, scale, fused operands, conversion, into the band's image
  auto columns = [&](int base, auto g) {
    constexpr int G = decltype(g)::value;
    v4i acc[G];
#pragma unroll
    for (int j = 0; j < G; ++j) acc[j] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      if (KT > 1 && kt >= a.k_tiles) break;
      const uint8_t* at = frag + kt * k_bytes + base * TILE16;
#pragma unroll
      for (int j = 0; j < G; ++j) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i*>(at + j * TILE16), xf[kt], acc[j], 0, 0, 0);
    }
    float v[G][4];
#pragma unroll
    for (int j = 0; j < G; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[j][i] = static_cast<float>(acc[j][i]) * scale;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const bool mul = p.binary[b].alg == ITEXHIP_BIN_MUL;
      // (the statements without instructions keep the compiler from computing more than one of the four and selecting)
      if (p.binary[b].stride_n == 0) {
        auto all = [&](auto f) {
          asm volatile("");
#pragma unroll
          for (int j = 0; j < G; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j][i] = f(v[j][i], uniform[b]);
        };
        if (mul) all([](float v, float o) { return v * o; });
        else all([](float v, float o) { return v + o; });
      } else {
        f4 o[G];
#pragma unroll
        for (int j = 0; j < G; ++j) o[j] = *reinterpret_cast<const f4*>(lds + a.operand_at[b] + ((base + j) * 16 + (lane >> 4) * 4) * 4);
        auto all = [&](auto f) {
          asm volatile("");
#pragma unroll
          for (int j = 0; j < G; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j][i] = f(v[j][i], o[j][i]);
        };
        if (mul) all([](float v, float o) { return v * o; });
        else all([](float v, float o) { return v + o; });
      }
    }
#pragma unroll
    for (int j = G - 1; j >= 0; --j) {
      uint8_t* to = mine + (base + j) * (16 * ESZ);
      auto write = [&](uint8_t* q, auto unaligned) {
        if constexpr (OUT_T == ITEXHIP_FLOAT) {
          using to_t = typename std::conditional<decltype(unaligned)::value, f4_any, f4>::type;
          *reinterpret_cast<to_t*>(q) = f4{v[j][0], v[j][1], v[j][2], v[j][3]};
        } else {
          using to_t = typename std::conditional<decltype(unaligned)::value, u2_any, u2>::type;
          *reinterpret_cast<to_t*>(q) = u2{f32x2_to_bits16<OUT_T>(v[j][0], v[j][1]), f32x2_to_bits16<OUT_T>(v[j][2], v[j][3])};
        }
      };
      write(to, std::false_type{});
      if (j == 0 && base == 0 && !a.whole_rows) {  // the first elements of a row stand behind the row above once more
        wave_sync();
        if ((lane >> 4) * 4 < VE && (lane & 15) > 0) write(to - a.pitch + N * ESZ, std::true_type{});
      }
    }
  };
  for (; band < band_end; band += kBandWaves) {
    const int m0 = band * kBand;
    turn_x(m0, image);
    // from the last tile, whose columns past N are garbage, to the first one, behind which a row's repeated elements go there
    int base = tiles16;
    if (tiles16 & 1) columns(base -= 1, std::integral_constant<int, 1>{});
    if (tiles16 & 2) columns(base -= 2, std::integral_constant<int, 2>{});
    while (base > 0) columns(base -= 4, std::integral_constant<int, 4>{});
    if (band + kBandWaves < band_end) load_x(m0 + kBandWaves * kBand);
    wave_sync();
    char* dst = out + (static_cast<int64_t>(bi) * M + m0) * N * ESZ;
    const int elements = min(M - m0, kBand) * N;
    if (a.whole_rows) {
      const int per_row = a.chunk / VE, live = min(a.chunk, N - n_first) / VE, pad = a.pitch - a.chunk * ESZ;
      char* to = dst + n_first * ESZ;
#pragma unroll 4
      for (int v = lane; v < min(M - m0, kBand) * per_row; v += 64) {
        const int row = fast_div(v, a.by_row), c = v - row * per_row;
        const v4i val = *reinterpret_cast<const v4i*>(image + v * 16 + row * pad);
        if (c < live) store16<STREAM>(to, row * (N * ESZ) + c * 16, val);
      }
    } else {
      const int head = min(static_cast<int>((16u - (static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst)) & 15u)) & 15u) / ESZ, elements);
      const int whole = (elements - head) / VE;
      // a wavefront's stores start on 128-byte lines: the first lanes may have nothing to do yet (four rows ahead of the image are
      // more than seven vectors)
      const int v0 = lane - static_cast<int>((static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst)) + head * ESZ) >> 4 & 7u);
      const int e0 = head + v0 * VE + 4 * N, row4 = fast_div(e0, a.by_row);
      int col = e0 - row4 * N, at = (row4 - 4) * a.pitch + col * ESZ;
      const int step = a.step_rows * a.pitch + a.step_cols * ESZ, wrap = a.pitch - N * ESZ;
      auto next = [&] {
        col += a.step_cols;
        at += step;
        if (col >= N) { col -= N; at += wrap; }
      };
      int v = v0;
      if (v < 0) { v += 64; next(); }
#pragma unroll 2
      for (; v < whole; v += 64) {
        const uint64_t* q = reinterpret_cast<const uint64_t*>(image + (at & ~7));
        const uint64_t d0 = q[0], d1 = q[1], d2 = q[2];
        const uint32_t w[5] = {at & 4 ? static_cast<uint32_t>(d0 >> 32) : static_cast<uint32_t>(d0), at & 4 ? static_cast<uint32_t>(d1) : static_cast<uint32_t>(d0 >> 32),
                               at & 4 ? static_cast<uint32_t>(d1 >> 32) : static_cast<uint32_t>(d1), at & 4 ? static_cast<uint32_t>(d2) : static_cast<uint32_t>(d1 >> 32),
                               at & 4 ? static_cast<uint32_t>(d2 >> 32) : static_cast<uint32_t>(d2)};
        v4i val;
        if constexpr (ESZ == 4) val = v4i{static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[2]), static_cast<int>(w[3])};
        else {
#pragma unroll
          for (int i = 0; i < 4; ++i) val[i] = static_cast<int>(__builtin_amdgcn_alignbyte(w[i + 1], w[i], at & 3));
        }
        store16<STREAM>(dst, head * ESZ + v * 16, val);
        next();
      }
      const int tail = elements - head - whole * VE;
      if (lane < head + tail) {
        const int e = lane < head ? lane : elements - tail + lane - head, r = fast_div(e, a.by_row);
        reinterpret_cast<elem_t*>(dst)[e] = *reinterpret_cast<const elem_t*>(image + r * a.pitch + (e - r * N) * ESZ);
      }
    }
    wave_sync();
  }
}

template <bool ADJ_Y, int NB, int OUT_T, int KT>
void launch_modes(const BandArgs& a, bool al, int lds, dim3 grid, const int8_t* x, const int8_t* y, char* out, hipStream_t st) {
  auto go = [&](auto mode) {
    auto kernel = qbmm_band_kernel<ADJ_Y, decltype(mode)::value, NB, OUT_T, KT>;
    static unsigned long long raised = 0;  // devices on which this kernel's LDS limit has been raised
    if (lds > 64 * 1024 && !device_bit(&raised, false) &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess)
      device_bit(&raised, true);
    kernel<<<grid, 64 * kBandWaves, lds, st>>>(a, x, y, out);
  };
  if constexpr (!ADJ_Y) {
    if (!al) return go(std::integral_constant<int, kAny>{});
  }
  go(std::integral_constant<int, kAligned>{});
}
template <bool ADJ_Y, int OUT_T>
void launch_ops(const BandArgs& a, bool al, int lds, dim3 grid, const int8_t* x, const int8_t* y, char* out, hipStream_t st) {
  auto go = [&](auto nb) {
    constexpr int NB = decltype(nb)::value;
    if (a.k_tiles == 1) launch_modes<ADJ_Y, NB, OUT_T, 1>(a, al, lds, grid, x, y, out, st);
    else launch_modes<ADJ_Y, NB, OUT_T, kMaxKTiles>(a, al, lds, grid, x, y, out, st);
  };
  if (a.p.n_binary == 0) go(std::integral_constant<int, 0>{});
  else if (a.p.n_binary == 1) go(std::integral_constant<int, 1>{});
  else go(std::integral_constant<int, 2>{});
}
template <int OUT_T>
void launch_out(const BandArgs& a, bool al, int lds, dim3 grid, const int8_t* x, const int8_t* y, char* out, hipStream_t st) {
  if (a.p.adj_y) launch_ops<true, OUT_T>(a, al, lds, grid, x, y, out, st);
  else launch_ops<false, OUT_T>(a, al, lds, grid, x, y, out, st);
}

}  // namespace

// Which calls come here, from products timed on both kernels (6900 of attention's two, 1 to 512 tokens, 8 to 4096 matrices, and 5100 around
// the lines; time of the bands over that of the tiles, in the middle; of those that come 2 and 5 % take over 1.05, at most 1.47).  `large`: the
// tiles would be those of 128 rows, at least 1024 of them, which compute past the edges of ragged matrices and hold few wavefronts per CU
// (aligned operands alone).  Everywhere while four workgroups (P.V: three) share the LDS of a CU; above that (wide results) it is 0.98 - 1.4,
// but for the second line.
// * y along k (Q.K^T), large: 16-bit results 0.70.
// * the same, 32-bit results whose rows are no multiple of 64 bytes, which the tiles write in pieces of lines: 0.65 with fused operands,
//   0.91 without them on up to 192 columns that are no whole 16-byte vectors a row (others 1.08); at any size of the images.  Rows of
//   whole 64-byte pieces up to 27 KB of LDS 0.68 (wider ones 1.10).
// * of those without operands, up to 224 MB of results (beyond, out of the memory-side cache, 0.36 - 1.3, 0.6), not: rows whose last 32 columns, a tile's
//   quadrant, are more than half full, K <= 96 0.53 - 1.42 (1.05; 182 x 32 x 182, 1053 times 36 -> 46 us), more than 176 columns 0.64 - 1.49 (1.08); nor,
//   at two workgroups a CU or one, more than 12 bands in a workgroup 0.43 - 1.42 (1.07), or a small last round 0.9 - 1.35 (1.1).  900 products: 34 over 1.05.
// * not where rows are no whole vectors: 16-bit results of up to 64 columns, one tile wide, 0.77 - 1.35 (1.08), or of one k tile and more than
//   256 rows by up to 128 columns 0.79 - 1.31 (1.27; 315 x 64 x 107, 3881 times 102 -> 133 us);  32-bit results of more than 192 columns without
//   operands 0.68 - 1.79 (1.21; 339 x 64 x 339, 265 times 32 -> 56), two workgroups or one on a CU that shift and store wide rows.
// * y transposed on the way (P.V), 16-bit results: large 0.73; K > 128, where a tile's k steps, one round trip each, are most of its
//   time, 0.84; K > 64 from 256 matrices on 0.92.  Below 0.95 - 1.07.
// * the same, 32-bit results: K > 192 0.92 (1.00 unaligned to 64 columns), K > 128 aligned 0.9, or up to 32 columns 0.78.  Below
//   1.0 - 1.2, large or not.
// * not where few tiles (two for a CU) of at most three k steps make a launch that the staging of more than 64 columns of y is a part of: over
//   96 columns, 64 with operands, 80 with 32-bit results 0.88 - 1.28 (1.09; 160 x 160 x 128, 12 times 4.4 -> 5.4);  a step more with operands and
//   an unaligned y of more than 80 columns 1.03 - 1.13;  nor with operands and unaligned rows on 49 to 64 columns, one tile wide, in many
//   tiles: 16-bit up to three k steps 0.84 - 1.27 (1.05; 107 x 107 x 64, 2085 times 14.6 -> 18.6), 32-bit up to five 0.97 - 1.20 (1.08).
// * not where the matrices are more than the device holds at once, of one tile of rows, a band for each wavefront behind the staging of a long y:
//   49 to 64 columns, K > 256 (32-bit results 192) 0.87 - 1.47 (1.18; 25 x 280 x 50, 3032 times 17.8 -> 23.3), 33 to 48 columns, K > 320 0.93 - 1.34
//   (1.05);  of two tiles of rows, 49 to 64 columns and K > 256 where the last round is a small one 0.96 - 1.31 (1.16; 95 x 304 x 50, 890 times 13.4 -> 17.6).
// * not 16-bit results whose rows are no whole vectors in few tiles: 49 to 64 columns, up to 1024 tiles of at most three k steps 0.91 - 1.21 (1.06), more
//   columns up to 256 tiles 0.94 - 1.26 (1.09; 102 x 208 x 100, 34 times 5.0 -> 5.9).
// Small launches of Q.K^T stay with the tiles (1.05 - 1.24): this kernel has a way through LDS more.
bool qbmm_band(const itexhip_bmm_params& p, int64_t batch, int mode_x, int mode_y, bool large, const int8_t* x, const int8_t* y, void* out,
               hipStream_t st) {
  if (p.adj_x || mode_x == kBytes || mode_y == kBytes || p.K < 16 || p.N < 16 || p.N > 2048 || p.K > kMaxKTiles * kTile) return false;
  if (p.M * p.K >= (1LL << 30) || p.M * p.N >= (1LL << 28)) return false;  // 32-bit offsets in a matrix
  for (int b = 0; b < p.n_binary; ++b)
    if (p.binary[b].stride_m != 0) return false;
  const int esz = p.out_type == ITEXHIP_FLOAT ? 4 : 2, ve = 16 / esz, N = static_cast<int>(p.N);
  const bool aligned_operands = mode_x == kAligned && mode_y == kAligned;
  if (p.adj_y ? !(large && aligned_operands)
              : esz == 2 ? !(large || p.K > 128 || (p.K > 64 && batch >= 256))
                         : !(p.K > 192 || (p.K > 128 && (aligned_operands || N <= 32)))) return false;
  BandArgs a;
  a.p = p;
  a.whole_rows = N * esz % 16 == 0 && aligned(out, 16);
  const bool operands = p.n_binary > 0, wide = esz == 4;
  // scores of fp32 without operands on ragged rows, whose tiles go out as fast where the results stay in the memory-side cache
  const bool bare = p.adj_y && wide && !operands && !a.whole_rows && batch * p.M * N * esz <= 224LL << 20;
  if (p.adj_y) {
    if (bare && (N - 1) % 32 >= 16 && (p.K <= 96 || N > 176)) return false;
    if (!a.whole_rows && (wide ? !operands && N > 192 : N <= 64 || (p.K <= 64 && p.M > 256 && N <= 128))) return false;
  } else {
    const int64_t tiles = batch * ((p.M + 63) / 64) * ((N + 63) / 64);
    if (tiles <= 512 && p.K <= 192 && N > (operands ? 64 : wide ? 80 : 96)) return false;
    if (operands && !aligned_operands &&
        (tiles > 2048 ? N > 48 && N <= 64 && p.K <= (wide ? 320 : 192) : !wide && tiles <= 256 && p.K <= 256 && N > 80)) return false;
    if (!wide && !a.whole_rows && N > 48 && ((tiles <= 256 && N > 64) || (tiles <= (N > 64 ? 512 : 1024) && p.K <= 192))) return false;
  }
  // rows of whole 64-byte pieces are cut into parts of at most 512 bytes, as even as they get (384 columns of fp32: 25.7 us whole,
  // 18.0 in three parts); the pieces of lines that parts of other rows would end in cost more than they give (216 columns of
  // fp32 in two parts 41 us, the tiles 23)
  a.chunk = N;
  if (a.whole_rows && N * esz % 64 == 0 && N * esz > 512) {
    const int n = (N * esz + 511) / 512, unit = 64 / esz;
    a.chunk = ((N + n - 1) / n + unit - 1) / unit * unit;
  }
  a.chunks = (N + a.chunk - 1) / a.chunk;
  a.rows16 = (a.chunk + 15) / 16 * 16;
  a.k_tiles = static_cast<int>((p.K + 63) / 64);
  // rows of the image start an odd number of 32-byte (64-byte, 32-bit results) pieces apart: the writes of 16 rows meet no bank twice
  const int piece = 16 * esz;
  a.pitch = ((a.chunk + (a.whole_rows ? 0 : ve)) * esz + piece - 1) / piece;
  a.pitch = (a.pitch + 1 - a.pitch % 2) * piece;
  a.band_bytes = std::max(kBand * a.pitch + 32, a.k_tiles * 1024);
  a.by_row = make_fast_div(a.whole_rows ? a.chunk / ve : N);
  a.step_rows = 64 * ve / N;
  a.step_cols = 64 * ve % N;
  a.bands_at = a.rows16 / 16 * a.k_tiles * tile16_bytes(p.adj_y != 0);
  for (int b = 0; b < p.n_binary; ++b) {
    a.operand_at[b] = a.bands_at;
    if (p.binary[b].stride_n != 0) a.bands_at += a.rows16 * 4;
  }
  const int lds = a.bands_at + kBandWaves * a.band_bytes;
  if (lds > 160 * 1024) return false;
  if (p.adj_y && esz == 4) {
    if (N * esz % 64 == 0 ? lds > 27 * 1024 : p.n_binary == 0 && a.whole_rows) return false;
  } else if (lds > (p.adj_y ? 40 : 52) * 1024) {
    return false;
  }
  // as many workgroups as the device holds at once (two to four on a CU), each with some of a matrix's bands: one that starts late
  // costs a round (Q.K^T over 197 tokens, bfloat16: 768 workgroups 12.3 us, 1536 of half as many bands 14.0)
  const int64_t resident = 256 * std::min(4, std::max(1, 160 * 1024 / lds));
  if (!p.adj_y && N > 32 && N <= 64 && batch > resident &&
      (p.M <= 64 ? p.K > (N <= 48 ? 320 : wide ? 192 : 256) : p.M <= 128 && N > 48 && p.K > 256 && batch * 10 <= resident * 13)) return false;
  a.batch = static_cast<uint32_t>(batch);
  a.bands = static_cast<int>((p.M + kBand - 1) / kBand);
  const int64_t want = std::min<int64_t>(std::max<int64_t>(1, resident / (batch * a.chunks)), (a.bands + kBandWaves - 1) / kBandWaves);
  a.bands_per_part = static_cast<int>((a.bands + want - 1) / want);
  if (bare && resident <= 512 && (a.bands_per_part > 12 || (batch > resident && batch * 10 < resident * 13))) return false;
  const int jobs = (a.bands + a.bands_per_part - 1) / a.bands_per_part * a.chunks;
  a.xcd_grid = batch % 8 == 0 || batch >= 64 ? 1 : 0;  // whole matrices per XCD: y is read into one L2
  if (jobs > 65535 || (a.xcd_grid ? (batch + 7) / 8 > 65535 : batch > 65535)) return false;
  // the dimensions that are missing have an extent of 1, the outermost ones
  const int missing = ITEXHIP_BMM_MAX_BATCH_DIMS - p.n_batch_dims;
  for (int d = 0; d < ITEXHIP_BMM_MAX_BATCH_DIMS; ++d) {
    const int from = d - missing;
    a.p.batch_dims[d] = from < 0 ? 1 : p.batch_dims[from];
    a.p.x_batch_stride[d] = from < 0 ? 0 : p.x_batch_stride[from];
    a.p.y_batch_stride[d] = from < 0 ? 0 : p.y_batch_stride[from];
    for (int b = 0; b < p.n_binary; ++b) a.p.binary[b].batch_stride[d] = from < 0 ? 0 : p.binary[b].batch_stride[from];
    a.by_dim[d] = make_fast_div(a.p.batch_dims[d]);
  }
  const dim3 grid = a.xcd_grid ? dim3(8, jobs, static_cast<unsigned>((batch + 7) / 8)) : dim3(jobs, static_cast<unsigned>(batch));
  note_kernel(kLastBands, a.chunks);
  char* o = static_cast<char*>(out);
  if (p.out_type == ITEXHIP_FLOAT) launch_out<ITEXHIP_FLOAT>(a, aligned_operands, lds, grid, x, y, o, st);
  else if (p.out_type == ITEXHIP_BFLOAT16) launch_out<ITEXHIP_BFLOAT16>(a, aligned_operands, lds, grid, x, y, o, st);
  else launch_out<ITEXHIP_HALF>(a, aligned_operands, lds, grid, x, y, o, st);
  return true;
}

}  // namespace itexhip
