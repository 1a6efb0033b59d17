// Quantized MatMul on operands as TensorFlow stores them: any K, no alignment, nothing prepacked.  It takes the problems
// whose K is not a multiple of 16 (the packed kernels move whole 16-byte pieces of an activation row).
//
// A workgroup owns a 64 x 64 output tile (32 x 32 where they are few, a kernel of its own below), whose K is walked in steps of 256: per step every thread fetches 64 bytes of the
// activations and 64 of the weight with 16-byte loads at whatever byte address they fall on (the hardware takes unaligned
// vector loads; two cache lines instead of one now and then), and puts them k-contiguous into LDS; a [K, N] weight is
// transposed on the way, 4 (k) x 16 (n) bytes per thread by byte permutes.  The long step is for latency: these problems
// have few tiles per CU, a step costs one round trip to L2 however long it is, and with 8 loads of 16 bytes per thread in
// flight during the previous step's MFMAs K = 1001 is 4 round trips, 2 where two groups of wavefronts share the steps.  n stays on the lanes of the accumulators
// (activation = first MFMA operand), so that stores are runs of 32 elements of an output row at any alignment and a lane
// needs the parameters of one channel per quadrant.
//
// Zero-point compensation needs the weight's column sums; they are dot products with ones of the words on their way into
// LDS (16 instructions per thread and step), added up across the workgroup once at the end.
//
// One thread per output element with byte loads is bound by its loads (two bytes per multiplication): 1000 x 1001 x 1000 with
// an fp32 result 399 -> 9.3 us, 43 times.  Short dot products of narrow results still go that way.
#include <algorithm>
#include <cmath>

#include "qgemm_common.hpp"

namespace itexhip {

namespace {

constexpr int kTileM = 64, kTileN = 64, kStepK = 256;
constexpr int kRow = kStepK + 16;  // LDS bytes per row: 16-byte fragment reads of 16 rows fall into 16 different bank groups

constexpr int kGroupLds = (kTileM + kTileN) * kRow;  // of a group of four wavefronts (the accumulators meet there as well)
static_assert(kGroupLds >= kTileM * kTileN * 4, "room for the accumulators");

// 16 bytes at base + off, any alignment.  A piece that would reach past the tensor's `end` is read from the last 16 bytes
// instead (the load is the same instruction for every lane; end >= 16) and moved into place by settle16, once it has
// arrived.
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));
__device__ __forceinline__ v4i fetch16(const uint8_t* __restrict__ base, int64_t off, int64_t end) {
  return *reinterpret_cast<const v4i_any*>(base + min(off, end - 16));
}
__device__ __forceinline__ v4i settle16(v4i v, int64_t off, int64_t end) {
  const int64_t over = off - (end - 16);
  // 0: in place; 16 and more: a piece that lies past the end as a whole, whose bytes are never used
  const uint32_t shift = over > 0 && over < 16 ? static_cast<uint32_t>(over) : 0;
  return shift_down(v, shift);
}

// the first `n` bytes of a piece (n < 16 cuts, n <= 0 clears)
__device__ __forceinline__ v4i keep_bytes(v4i v, int n) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int left = n - 4 * i;
    const uint32_t mask = left >= 4 ? 0xffffffffu : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
    v[i] = static_cast<int>(static_cast<uint32_t>(v[i]) & mask);
  }
  return v;
}

// Where byte k of weight column n lives in LDS.  The four 16-column groups that a wavefront of the transposing writer
// serves at once would meet in the same banks (16 rows are a multiple of all of them apart): each group keeps its 64-byte
// quarters of a 256-byte span in another order.
__device__ __forceinline__ int w_offset(int n, int k) { return n * kRow + (k ^ (((n >> 4) & 3) << 6)); }

// column 4 c + j of four rows' bytes -> v[j]
__device__ __forceinline__ void transpose_bytes(const v4i (&rows)[4], int c, uint32_t (&v)[4]) {
  const uint32_t w[4] = {static_cast<uint32_t>(rows[0][c]), static_cast<uint32_t>(rows[1][c]), static_cast<uint32_t>(rows[2][c]),
                         static_cast<uint32_t>(rows[3][c])};
  transpose_4x4(w, v);
}

template <int ALG, int COUNT>
__device__ __forceinline__ void apply_all(const itexhip_eltwise& elt, float (&v)[COUNT]) {
  itexhip_eltwise e = elt;
  e.alg = ALG;  // known here: apply_eltwise folds to one case
#pragma unroll
  for (int i = 0; i < COUNT; ++i) v[i] = apply_eltwise(e, v[i]);
}

// the post-ops on COUNT results; index(i): where result i stands in the output (the summand's element)
template <int COUNT, typename Index>
__device__ __forceinline__ void apply_chain(const EpilogueArgs& e, float (&v)[COUNT], Index&& index) {
  for (int k = 0; k < e.n_eltwise; ++k) {
    const itexhip_eltwise& elt = e.elt[k];
    switch (elt.alg) {
      case ITEXHIP_ELT_SUM:
#pragma unroll
        for (int i = 0; i < COUNT; ++i) v[i] = v[i] + elt.alpha * load_addend(e, index(i));
        break;
      case ITEXHIP_ELT_RELU: apply_all<ITEXHIP_ELT_RELU>(elt, v); break;
      case ITEXHIP_ELT_CLIP: apply_all<ITEXHIP_ELT_CLIP>(elt, v); break;
      case ITEXHIP_ELT_LINEAR: apply_all<ITEXHIP_ELT_LINEAR>(elt, v); break;
      case ITEXHIP_ELT_GELU_TANH: apply_all<ITEXHIP_ELT_GELU_TANH>(elt, v); break;
      case ITEXHIP_ELT_GELU_ERF: apply_all<ITEXHIP_ELT_GELU_ERF>(elt, v); break;
      case ITEXHIP_ELT_ELU: apply_all<ITEXHIP_ELT_ELU>(elt, v); break;
      case ITEXHIP_ELT_LOGISTIC: apply_all<ITEXHIP_ELT_LOGISTIC>(elt, v); break;
      case ITEXHIP_ELT_TANH: apply_all<ITEXHIP_ELT_TANH>(elt, v); break;
      case ITEXHIP_ELT_SWISH: apply_all<ITEXHIP_ELT_SWISH>(elt, v); break;
      case ITEXHIP_ELT_MISH: apply_all<ITEXHIP_ELT_MISH>(elt, v); break;
      default: break;
    }
  }
}

// SPLIT groups of four wavefronts share a tile: group g takes the K steps g, g + SPLIT, ... in LDS of its own, so that the
// first SPLIT steps' loads are all in flight at once, and the groups' accumulators meet in LDS at the end, where each group
// finishes 16 / SPLIT of a lane's 16 rows.  A launch of few tiles is a chain of latencies (start, one round trip per step,
// parameters, stores: 6 us without its steps, 1.2 per step), which two groups shorten; four (128 registers, 1024 threads to
// start) are slower than two up to K = 2000.
template <int OUT_T, bool TRANS, int SPLIT>
__global__ __launch_bounds__(256 * SPLIT) void qmatmul_unpacked_kernel(const uint8_t* __restrict__ a, uint32_t a_xor,
                                                                const uint8_t* __restrict__ w, int M, int K, int N,
                                                                int tiles_n, int tiles, EpilogueArgs e, void* __restrict__ out) {
  // per group its rows and columns, then the column sums (one group: at addresses that the compiler knows)
  extern __shared__ __attribute__((aligned(16))) uint8_t dynamic_lds[];
  uint8_t* lds = dynamic_lds;
  if constexpr (SPLIT == 1) {
    __shared__ __attribute__((aligned(16))) uint8_t fixed[kGroupLds + 4 * kTileN];
    lds = fixed;
  }
  const int t = threadIdx.x & 255, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int group = SPLIT == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  uint8_t* const as = lds + group * kGroupLds;
  uint8_t* const ws = as + kTileM * kRow;
  int* const colsum = reinterpret_cast<int*>(lds + SPLIT * kGroupLds);
  // consecutive workgroup ids go round the 8 XCDs: give each of them a contiguous run of tiles (n fastest), whose
  // activation rows its L2 then fetches once
  const int per_xcd = (tiles + 7) / 8;
  const int tile = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || tile >= tiles) return;  // whole workgroup
  const int tm = tile / tiles_n;
  const int m0 = tm * kTileM, n0 = (tile - tm * tiles_n) * kTileN;
  const int64_t a_end = static_cast<int64_t>(M) * K, w_end = static_cast<int64_t>(K) * N;
  const bool want_sums = e.comp_mul != 0 || e.prep.input_mode == ITEXHIP_MIN_FIRST;
  if (threadIdx.x < kTileN) colsum[threadIdx.x] = 0;

  // fetch roles: rows (of the activations, or of an [N, K] weight): row t / 16 + 16 h, piece t % 16
  //              [K, N] weight: 4 k rows from 4 * (t / 4), 16 columns from 16 * (t % 4)
  const int frow = t >> 4, fpiece = (t & 15) * 16;
  const int kb = t >> 2, nb = (t & 3) * 16;
  v4i fa[4], fw[4];
  int sums[TRANS ? 4 : 16];
#pragma unroll
  for (int i = 0; i < (TRANS ? 4 : 16); ++i) sums[i] = 0;

  auto a_off = [&](int h, int k0) {  // rows past M repeat the last one (their results are not stored)
    return static_cast<int64_t>(min(m0 + frow + 16 * h, M - 1)) * K + k0 + fpiece;
  };
  auto w_off = [&](int h, int k0) {
    if constexpr (TRANS) return static_cast<int64_t>(min(n0 + frow + 16 * h, N - 1)) * K + k0 + fpiece;
    else return static_cast<int64_t>(k0 + kb * 4 + h) * N + n0 + nb;
  };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int h = 0; h < 4; ++h) fa[h] = fetch16(a, a_off(h, k0), a_end);
#pragma unroll
    for (int h = 0; h < 4; ++h) fw[h] = fetch16(w, w_off(h, k0), w_end);
  };
  // What lies past K is whatever follows in the activations and zero in the weight.  Pieces that reach past a tensor's end
  // only occur in the last rows of the last step: the whole workgroup tests for that once per step.
  auto put = [&](int k0) {
    const bool last = k0 + kStepK + 16 > K;
    if (last) {
      if (m0 + kTileM + 16 > M) {
#pragma unroll
        for (int h = 0; h < 4; ++h) fa[h] = settle16(fa[h], a_off(h, k0), a_end);
      }
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        fw[h] = settle16(fw[h], w_off(h, k0), w_end);
        if constexpr (TRANS) fw[h] = keep_bytes(fw[h], K - k0 - fpiece);
        else if (k0 + kb * 4 + h >= K) fw[h] = v4i{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      v4i v = fa[h];
      v.x ^= a_xor; v.y ^= a_xor; v.z ^= a_xor; v.w ^= a_xor;
      *reinterpret_cast<v4i*>(as + (frow + 16 * h) * kRow + fpiece) = v;
    }
    if constexpr (TRANS) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const v4i v = fw[h];
        *reinterpret_cast<v4i*>(ws + w_offset(frow + 16 * h, fpiece)) = v;
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[h] = __builtin_amdgcn_sdot4(v[i], 0x01010101, sums[h], false);
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {  // columns nb + 4 c .. + 3: a 4 x 4 byte transpose in two rounds of permutes
        uint32_t v[4];
        transpose_bytes(fw, c, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          *reinterpret_cast<uint32_t*>(ws + w_offset(nb + 4 * c + j, kb * 4)) = v[j];
          sums[4 * c + j] = __builtin_amdgcn_sdot4(static_cast<int>(v[j]), 0x01010101, sums[4 * c + j], false);
        }
      }
    }
  };

  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  v16i acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0;
  if (group * kStepK < K) fetch(group * kStepK);
  // the channel this lane finishes; its parameters travel under the K loop, behind the first step's operands
  // (ahead of them, their pointers' way out of the kernel's arguments stood in front: 1000 x 1001 x 1000 9.7 -> 9.3 us, calls one
  // after another on a stream; the same in a graph, 9.8)
  const int n = n0 + wn + (lane & 31);
  RawChannel raw = load_raw_channel(e, min(n, N - 1), N);
  for (int round = 0; round < K; round += SPLIT * kStepK) {
    const int k0 = round + group * kStepK;  // a group may have no step in the last round
    if (k0 < K) put(k0);
    __syncthreads();
    if (k0 + SPLIT * kStepK < K) fetch(k0 + SPLIT * kStepK);
    auto multiply = [&](int kk) {
      const int k = kk + (lane >> 5) * 16;
      const v4i x = *reinterpret_cast<const v4i*>(as + (wm + (lane & 31)) * kRow + k);
      const v4i y = *reinterpret_cast<const v4i*>(ws + w_offset(wn + (lane & 31), k));
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, y, acc, 0, 0, 0);
    };
    if (k0 + kStepK <= K) {
#pragma unroll
      for (int kk = 0; kk < kStepK; kk += 32) multiply(kk);
    } else {
      for (int kk = 0; k0 + kk < K; kk += 32) multiply(kk);
    }
    __syncthreads();
  }
  if (want_sums) {
    if constexpr (TRANS) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) sums[h] += __shfl_xor(sums[h], d, 64);
        if ((t & 15) == 0) {
          if constexpr (SPLIT == 1) colsum[frow + 16 * h] = sums[h];
          else atomicAdd(&colsum[frow + 16 * h], sums[h]);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {  // over the 4 lanes of a row of 16 that hold these columns, then across rows and wavefronts
        sums[i] += __shfl_xor(sums[i], 4, 64);
        sums[i] += __shfl_xor(sums[i], 8, 64);
        if ((lane & 12) == 0) atomicAdd(&colsum[nb + i], sums[i]);
      }
    }
  }
  constexpr int kPer = 16 / SPLIT;  // rows of a lane that this group finishes, from `first` on
  const int first = group * kPer;
  int sum[kPer];
  if constexpr (SPLIT == 1) {
    if (want_sums) __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) sum[i] = acc[i];
  } else {
    // (the loop's last barrier: no wavefront reads its operands any more)
    int* const mine = reinterpret_cast<int*>(as) + wave * 16 * 64 + lane;
#pragma unroll
    for (int i = 0; i < 16; ++i) mine[i * 64] = acc[i];
    __syncthreads();
    const int* src = reinterpret_cast<const int*>(lds) + (wave * 16 + first) * 64 + lane;
#pragma unroll
    for (int i = 0; i < kPer; ++i) sum[i] = 0;
#pragma unroll
    for (int g = 0; g < SPLIT; ++g)
#pragma unroll
      for (int i = 0; i < kPer; ++i) sum[i] += src[g * (kGroupLds / 4) + i * 64];
  }
  if (n >= N) return;
  raw.colsum = colsum[wn + (lane & 31)];
  int comp;
  float scale, bias;
  finish_channel(e, raw, &comp, &scale, &bias);
  // accumulator i of a lane: row (i / 4) * 8 + (lane / 32) * 4 + i % 4, column lane % 32 of the quadrant
  const int mrow = m0 + wm + (lane >> 5) * 4;
  auto row_of = [&](int i) { return mrow + ((first + i) >> 2) * 8 + ((first + i) & 3); };
  float v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    v[i] = static_cast<float>(sum[i] + comp) * scale;  // scale 1.0f when the node has no output scale (exact)
    v[i] = v[i] + bias;
  }
  apply_chain(e, v, [&](int i) { return static_cast<int64_t>(min(row_of(i), M - 1)) * N + n; });
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int m = row_of(i);
    if (m < M) store_output<OUT_T>(out, static_cast<int64_t>(m) * N + n, v[i]);
  }
}

// Few tiles and a [K, N] weight: 32 x 32 results per workgroup, whose WAVES wavefronts take 128 k each in turn and share nothing
// until their accumulators meet in LDS at the end.  The 64 x 64 tiles are bound by their loads there: one at an odd byte address
// is served a lane per clock however its lanes lie.  So here the activations come straight as MFMA operands, row by lane, and
// lanes without a row or a column load nothing; the weight is transposed through LDS that belongs to the wavefront, and its
// column sums are a second product, with ones.  A CU has half the loads to serve, four times as many CUs share them, and up to
// 128 WAVES k all are in flight at once.  us, 64 x 64 tiles -> these: 10 x 943 x 9 9.7 -> 5.3, 23 x 961 x 364 9.1 -> 5.9, 300 x 511 x 300
// 7.3 -> 5.9, 200 x 901 x 1000 9.2 -> 7.4, 64 x 4001 x 64 19.3 -> 14.6, 10 x 137 x 28 6.8 -> 4.3.
constexpr int kFew = 32, kFewK = 128, kFewRow = kFewK + 16;
template <int OUT_T, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void qmatmul_unpacked_few_kernel(const uint8_t* __restrict__ a, uint32_t a_xor,
                                                                              const uint8_t* __restrict__ w, int M, int K, int N,
                                                                              int tiles_n, int tiles, EpilogueArgs e, void* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[WAVES][kFew * kFewRow];  // the wavefront's weight, then its accumulators
  __shared__ int colsums[WAVES][kFew];
  static_assert(kFew * kFewRow >= kFew * kFew * 4, "room for the accumulators");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int l32 = lane & 31, half = lane >> 5;
  // contiguous runs of tiles for the 8 XCDs, as above
  const int per_xcd = (tiles + 7) / 8;
  const int tile = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || tile >= tiles) return;  // whole workgroup
  const int tm = tile / tiles_n;
  const int m0 = tm * kFew, n0 = (tile - tm * tiles_n) * kFew;
  const int64_t a_end = static_cast<int64_t>(M) * K, w_end = static_cast<int64_t>(K) * N;
  const bool want_sums = e.comp_mul != 0 || e.prep.input_mode == ITEXHIP_MIN_FIRST;
  uint8_t* const ws = lds[wave];
  const int kb = (lane >> 1) * 4, nb = (lane & 1) * 16;  // [K, N] weight: 4 rows of 16 columns
  v16i acc, sums;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = sums[i] = 0;
  v4i fa[4], fw[4];
  const bool row_here = m0 + l32 < M, column_here = n0 + nb < N;
  auto a_off = [&](int c, int k0) { return static_cast<int64_t>(m0 + l32) * K + k0 + c * 32 + half * 16; };
  auto w_off = [&](int c, int k0) { return static_cast<int64_t>(k0 + kb + c) * N + n0 + nb; };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int c = 0; c < 4; ++c) fa[c] = fw[c] = v4i{0, 0, 0, 0};
    if (row_here) {
#pragma unroll
      for (int c = 0; c < 4; ++c) fa[c] = fetch16(a, a_off(c, k0), a_end);
    }
    if (column_here) {
#pragma unroll
      for (int c = 0; c < 4; ++c) fw[c] = fetch16(w, w_off(c, k0), w_end);
    }
  };
  int k0 = wave * kFewK;
  if (k0 < K) fetch(k0);
  const int n = n0 + l32;
  RawChannel raw = load_raw_channel(e, min(n, N - 1), N);  // travels behind the operands
  for (; k0 < K; k0 += WAVES * kFewK) {
    if (k0 + kFewK + 16 > K) {  // pieces past a tensor's end; what lies past K is zero in the weight (see the other kernel)
      if (m0 + kFew + 16 > M) {
#pragma unroll
        for (int c = 0; c < 4; ++c) fa[c] = settle16(fa[c], a_off(c, k0), a_end);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        fw[c] = settle16(fw[c], w_off(c, k0), w_end);
        if (k0 + kb + c >= K) fw[c] = v4i{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      uint32_t v[4];
      transpose_bytes(fw, c, v);
      // (the 16 columns of the other lanes would fall into the same banks: they keep their halves of a row the other way round)
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<uint32_t*>(ws + (nb + 4 * c + j) * kFewRow + (kb ^ (nb << 2))) = v[j];
    }
    v4i x[4], y[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      x[c] = fa[c];
      x[c].x ^= a_xor; x[c].y ^= a_xor; x[c].z ^= a_xor; x[c].w ^= a_xor;
      y[c] = *reinterpret_cast<const v4i*>(ws + l32 * kFewRow + ((c * 32 + half * 16) ^ ((l32 & 16) << 2)));
    }
    if (k0 + WAVES * kFewK < K) fetch(k0 + WAVES * kFewK);
#pragma unroll
    for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[c], y[c], acc, 0, 0, 0);
    if (want_sums) {
      const v4i ones = v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
      for (int c = 0; c < 4; ++c) sums = __builtin_amdgcn_mfma_i32_32x32x32_i8(ones, y[c], sums, 0, 0, 0);
    }
  }
  int* const mine = reinterpret_cast<int*>(ws) + lane;
#pragma unroll
  for (int i = 0; i < 16; ++i) mine[i * 64] = acc[i];
  if (half == 0) colsums[wave][l32] = sums[0];
  __syncthreads();
  constexpr int kPer = 16 / WAVES;  // results of a lane that this wavefront finishes, from `first` on
  const int first = wave * kPer;
  int sum[kPer];
  raw.colsum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) sum[i] = 0;
#pragma unroll
  for (int g = 0; g < WAVES; ++g) {
    raw.colsum += colsums[g][l32];
#pragma unroll
    for (int i = 0; i < kPer; ++i) sum[i] += reinterpret_cast<const int*>(lds[g])[(first + i) * 64 + lane];
  }
  if (n >= N) return;
  int comp;
  float scale, bias;
  finish_channel(e, raw, &comp, &scale, &bias);
  // accumulator i of a lane: row (i / 4) * 8 + (lane / 32) * 4 + i % 4, column lane % 32
  auto row_of = [&](int i) { return m0 + half * 4 + ((first + i) >> 2) * 8 + ((first + i) & 3); };
  float v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    v[i] = static_cast<float>(sum[i] + comp) * scale;
    v[i] = v[i] + bias;
  }
  apply_chain(e, v, [&](int i) { return static_cast<int64_t>(min(row_of(i), M - 1)) * N + n; });
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int m = row_of(i);
    if (m < M) store_output<OUT_T>(out, static_cast<int64_t>(m) * N + n, v[i]);
  }
}

// One thread per output element, from `first` on (in_pieces; a loop over the outputs in here costs 20 %).  Takes what the tile kernel cannot (an operand of fewer
// than 16 bytes in all, too many tiles for a launch) and short dot products of narrow results, see one_output_per_thread.
template <int OUT_T>
__global__ __launch_bounds__(256) void qmatmul_tiny_kernel(const uint8_t* __restrict__ a, int a_is_u8,
                                                            const int8_t* __restrict__ w, int transpose_b,
                                                            int M, int K, int N, EpilogueArgs e,
                                                            void* __restrict__ out, int64_t first) {
  const int64_t idx = first + static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= static_cast<int64_t>(M) * N) return;
  const int m = static_cast<int>(idx / N), n = static_cast<int>(idx % N);
  int acc = 0, wsum = 0;
  for (int k = 0; k < K; ++k) {
    const int av = a_is_u8 ? static_cast<int>(a[static_cast<int64_t>(m) * K + k])
                           : static_cast<int>(reinterpret_cast<const int8_t*>(a)[static_cast<int64_t>(m) * K + k]);
    const int wv = transpose_b ? w[static_cast<int64_t>(n) * K + k] : w[static_cast<int64_t>(k) * N + n];
    acc += av * wv;
    wsum += wv;
  }
  const int jb = (e.nb == N) ? n : 0;
  const ChannelScaleBias c = channel_scale_bias(e.prep, e.min_b[jb], e.max_b[jb], e.min_b[0], e.max_b[0],
                                                bias_entry(e.prep, e.bias, n), wsum);
  float v = static_cast<float>(acc);
  if (e.n_scales > 0) v = v * c.scale;
  v = v + c.bias;
  for (int k = 0; k < e.n_eltwise; ++k) {
    if (e.elt[k].alg == ITEXHIP_ELT_SUM) v = v + e.elt[k].alpha * load_addend(e, idx);
    else v = apply_eltwise(e.elt[k], v);
  }
  store_output<OUT_T>(out, idx, v);
}

// Short dot products, and narrow results: a tile of the other kernel costs the same whether one of its rows or columns exists or
// all 64 do, and however much of its first K step.  Times in us as both kernels measured (17000 sizes of 1 to 200000 rows and
// columns, K of 1 to 300).  A thread per output: the latency of its dot product, 2.4 + 0.071 K (0.105 K beyond 64 columns), or,
// where the outputs fill the chip, 2 and 1e-6 of 3.4 + 0.26 K per output, more per k where a wavefront's 64 outputs touch many
// rows (few columns, rows that share no lines) and where the weight is past 2 MB; in between the two join.  Tiles: 3.4 + 0.011
// each, at least 5.8, per further K step half of that more and 0.9 (one group of wavefronts; two are shorter, but from the second
// step on a thread's dot product alone takes 20).  The choice is 0.2 % above the faster kernel in the mean and
// takes the slower one where it costs more than 10 % for 84 of the sizes (up to twice: 122975 x 107 x 1 45 for 23).
// Per output / tiles: 100000 x 17 x 1 4.8 / 20.7, 1 x 17 x 100000 5.3 / 20.3, 1000000 x 9 x 16 99 / 143, 8 x 9 x 8 3.6 / 6.0,
// 270 x 9 x 1413 4.6 / 6.4, 13 x 19 x 36455 6.6 / 11.2; 100000 x 65 x 10 57 / 21, 84678 x 32 x 11 30 / 15, 1000 x 17 x 1000
// 11.3 / 6.8.
bool one_output_per_thread(int64_t M, int64_t K, int64_t N, int64_t tiles) {
  const double k = static_cast<double>(K), n = static_cast<double>(N), outputs = static_cast<double>(M) * n;
  const double per_k = 0.26 + (K * N > 1 << 21 ? 0.45 : 0.0) + std::min(1.3, k / 24.0) * 2.2 / (n + 1.3);
  const double latency = 2.4 + (N <= 64 ? 0.071 : 0.105) * k, filled = 2.0 + 1e-6 * outputs * (3.4 + per_k * k);
  const double threads = std::cbrt(latency * latency * latency + filled * filled * filled);
  const double steps = static_cast<double>((K + kStepK - 1) / kStepK);
  return threads < std::max(5.8, 3.4 + 0.0055 * (1.0 + steps) * static_cast<double>(tiles)) + 0.9 * (steps - 1.0);
}

template <int OUT_T, bool TRANS, int SPLIT>
int launch_tiles(unsigned grid, const uint8_t* a, uint32_t a_xor, const uint8_t* w, int M, int K, int N, int tiles_n, int tiles,
                 const EpilogueArgs& e, void* out, hipStream_t st) {
  auto kern = qmatmul_unpacked_kernel<OUT_T, TRANS, SPLIT>;
  constexpr int kLds = SPLIT == 1 ? 0 : SPLIT * kGroupLds + 4 * kTileN;  // dynamic
  static unsigned long long attr_done = 0;  // devices on which this instantiation's attribute is set
  if (kLds > 64 * 1024 && !device_bit(&attr_done, false)) {
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (err != hipSuccess) return hip_fail(err, "hipFuncSetAttribute(qmatmul_unpacked_kernel)");
    device_bit(&attr_done, true);
  }
  note_kernel(kLastUnpacked, SPLIT);
  kern<<<grid, 256 * SPLIT, kLds, st>>>(a, a_xor, w, M, K, N, tiles_n, tiles, e, out);
  return ITEXHIP_OK;
}

template <int OUT_T>
int launch(const uint8_t* a, uint32_t a_xor, const uint8_t* w, int transpose_b, int M, int K, int N, int tiles_n, int tiles,
            const EpilogueArgs& e, void* out, hipStream_t st) {
  const bool forced = __atomic_load_n(&g_forced_tile_shape[0], __ATOMIC_RELAXED) >= 0;  // tests ask for the tile kernel
  if (tiles == 0 || static_cast<int64_t>(M) * K < 16 || static_cast<int64_t>(K) * N < 16 || (!forced && one_output_per_thread(M, K, N, tiles))) {
    note_kernel(kLastPerOutput, 0);
    in_pieces(0, static_cast<int64_t>(M) * N, [&](int64_t first, int64_t end) {
      qmatmul_tiny_kernel<OUT_T><<<static_cast<unsigned>((end - first + 255) / 256), 256, 0, st>>>(
          a, a_xor != 0, reinterpret_cast<const int8_t*>(w), transpose_b, M, K, N, e, out, first);
    });
    return ITEXHIP_OK;
  }
  const unsigned grid = static_cast<unsigned>((tiles + 7) / 8 * 8);  // whole runs for the 8 XCDs
  // Two groups per tile as long as every tile has a CU to itself, with one K step only where the weight is [N, K] (it is put
  // into LDS as it is); beyond that a CU runs two workgroups of one group and hides one's waits behind the other, where one
  // workgroup of two groups is all that its registers hold.  One group / two, us: 1000 x 1001 x 1000 (256 tiles) 11.0 / 9.7,
  // 200 x 901 x 1000 10.2 / 8.9, 300 x 511 x 300 8.1 / 7.3; 2000 x 301 x 1000 (512 tiles) 9.4 / 13.0.  Two / one over 1500 sizes of
  // one step: [N, K] 0.93 - 1.07 (0.99 in the middle), [K, N] 0.96 - 1.10 (1.02: 3 x 43 x 68 5.6 / 6.1); of more steps 0.81 - 0.99.
  const bool split = tiles <= 256 && (transpose_b || K > kStepK);
  // 32 x 32 tiles, time over the kernel that took these calls (1400 sizes of up to 4000 rows, columns and k): up to 256 of them 0.35 - 1.0
  // (0.68 in the middle), 257 - 512 with K <= 512 0.73 - 0.94 (0.78), with more 0.84 - 1.16 (not there), more tiles 1.05 - 2.
  const int64_t few_n = (N + kFew - 1) / kFew, few = (static_cast<int64_t>(M) + kFew - 1) / kFew * few_n;
  if (!transpose_b && !forced && (few <= 256 || (few <= 512 && K <= 512))) {
#define FEW(WAVES)                                                                                                               \
  note_kernel(kLastUnpacked, WAVES / 4);                                                                                         \
  qmatmul_unpacked_few_kernel<OUT_T, WAVES><<<static_cast<unsigned>((few + 7) / 8 * 8), 64 * WAVES, 0, st>>>(                     \
      a, a_xor, w, M, K, N, static_cast<int>(few_n), static_cast<int>(few), e, out)
    if (K > 4 * kFewK) {
      FEW(8);
    } else {
      FEW(4);
    }
#undef FEW
    return ITEXHIP_OK;
  }
#define TILES(S) (transpose_b ? launch_tiles<OUT_T, true, S>(grid, a, a_xor, w, M, K, N, tiles_n, tiles, e, out, st) \
                              : launch_tiles<OUT_T, false, S>(grid, a, a_xor, w, M, K, N, tiles_n, tiles, e, out, st))
  return split ? TILES(2) : TILES(1);
#undef TILES
}

}  // namespace

// M, N > 0; `e` is a fused epilogue (the kernel derives scale and bias of a channel itself) without column sums.
int launch_unpacked(const void* a, int a_type, const int8_t* w, int transpose_b, int64_t M, int64_t K, int64_t N,
                    const EpilogueArgs& e, int out_type, void* out, hipStream_t st, const char* who) {
  const int64_t tiles_m = (M + kTileM - 1) / kTileM, tiles_n = (N + kTileN - 1) / kTileN;
  // a launch has fewer than 2^32 threads; a result of more tiles than that allows goes one thread per output element
  const bool many_tiles = tiles_m * tiles_n >= (1LL << 24) - 8;
  const uint8_t* ap = static_cast<const uint8_t*>(a);
  const uint8_t* wp = reinterpret_cast<const uint8_t*>(w);
  const uint32_t a_xor = a_type == ITEXHIP_QUINT8 ? 0x80808080u : 0u;
  const int Mi = static_cast<int>(M), Ki = static_cast<int>(K), Ni = static_cast<int>(N);
  const int tn = static_cast<int>(tiles_n), tiles = many_tiles ? 0 : static_cast<int>(tiles_m * tiles_n);
  int rc;
  switch (out_type) {
    case ITEXHIP_FLOAT: rc = launch<ITEXHIP_FLOAT>(ap, a_xor, wp, transpose_b, Mi, Ki, Ni, tn, tiles, e, out, st); break;
    case ITEXHIP_BFLOAT16: rc = launch<ITEXHIP_BFLOAT16>(ap, a_xor, wp, transpose_b, Mi, Ki, Ni, tn, tiles, e, out, st); break;
    case ITEXHIP_HALF: rc = launch<ITEXHIP_HALF>(ap, a_xor, wp, transpose_b, Mi, Ki, Ni, tn, tiles, e, out, st); break;
    case ITEXHIP_QINT32: rc = launch<ITEXHIP_QINT32>(ap, a_xor, wp, transpose_b, Mi, Ki, Ni, tn, tiles, e, out, st); break;
    case ITEXHIP_QINT8: rc = launch<ITEXHIP_QINT8>(ap, a_xor, wp, transpose_b, Mi, Ki, Ni, tn, tiles, e, out, st); break;
    default: rc = launch<ITEXHIP_QUINT8>(ap, a_xor, wp, transpose_b, Mi, Ki, Ni, tn, tiles, e, out, st); break;
  }
  if (rc != ITEXHIP_OK) return rc;
  ITEXHIP_CHECK_LAUNCH(who);
  return ITEXHIP_OK;
}

}  // namespace itexhip
