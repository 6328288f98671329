// Kernels around the attention path of the serving loop, for gfx950:
//   * add_rmsnorm       -- RMSNorm with the residual add fused (src/layers/layernorm.py:11-28)
//   * silu_and_mul      -- SiluAndMul (src/layers/activation.py:6-10)
//   * lm_head_greedy    -- logits = x W^T (src/layers/llm_head.py:60-64) followed by a greedy
//                          argmax, without writing the logits
//
// Rounding points follow the reference. The norms compute in fp32 and round the output
// (and the new residual) to bf16. SiluAndMul runs under torch.compile, which upcasts both
// halves, computes silu(x) * y in fp32 and rounds once. The LM head's logits are bf16 in
// the reference (F.linear on bf16 operands); the greedy choice here compares the fp32 dot
// products after rounding them to bf16 and keeps the lowest vocabulary index among equal
// maxima, which is what argmax over the bf16 logits returns.
#include <algorithm>

#include "common.h"

namespace pk {
namespace {

__device__ __forceinline__ float round_to_bf16(float f) {
  return __uint_as_float((uint32_t)f32_to_bf16(f) << 16);
}

// ---------------------------------------------------------------- add + RMSNorm ---------

constexpr int kNormThreads = 128;

// One work-group per row; each thread owns 8 consecutive elements (hidden <= 8 * 128 * 4).
// out = bf16(w * (s * rsqrt(mean(s^2) + eps))) with s = x (+ residual) in fp32;
// residual_out = bf16(s) when a residual is given (layernorm.py:24-28), else untouched.
template <int kVecs>
__global__ __launch_bounds__(kNormThreads) void add_rmsnorm_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* residual, int64_t res_stride,
    const uint16_t* __restrict__ weight, float eps, int32_t hidden, uint16_t* out, int64_t out_stride,
    uint16_t* residual_out, int64_t res_out_stride) {
  const int64_t row = blockIdx.x;
  // x, residual and weight loads all go out before any of them is used (one round of loads)
  uint4 xv[kVecs], rv[kVecs], wv[kVecs];
#pragma unroll
  for (int j = 0; j < kVecs; ++j) {
    const int col = (j * kNormThreads + threadIdx.x) * 8;
    if (col < hidden) {
      xv[j] = *reinterpret_cast<const uint4*>(x + row * x_stride + col);
      rv[j] = residual != nullptr ? *reinterpret_cast<const uint4*>(residual + row * res_stride + col)
                                  : make_uint4(0, 0, 0, 0);
      wv[j] = *reinterpret_cast<const uint4*>(weight + col);
    }
  }
  float v[kVecs][8];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < kVecs; ++j) {
    const int col = (j * kNormThreads + threadIdx.x) * 8;
    if (col < hidden) {
      const uint32_t ww[4] = {xv[j].x, xv[j].y, xv[j].z, xv[j].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[j][2 * e] = bf16_lo(ww[e]);
        v[j][2 * e + 1] = bf16_hi(ww[e]);
      }
      if (residual != nullptr) {
        const uint32_t rr[4] = {rv[j].x, rv[j].y, rv[j].z, rv[j].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[j][2 * e] += bf16_lo(rr[e]);
          v[j][2 * e + 1] += bf16_hi(rr[e]);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[j][e], v[j][e], ss);
    }
  }
  for (int m = kWave / 2; m >= 1; m >>= 1) ss += xor_shfl(ss, m);
  __shared__ float part[kNormThreads / kWave];
  if ((threadIdx.x & (kWave - 1)) == 0) part[threadIdx.x / kWave] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < kNormThreads / kWave; ++i) tot += part[i];
  const float rs = 1.0f / __builtin_sqrtf(tot / (float)hidden + eps);
#pragma unroll
  for (int j = 0; j < kVecs; ++j) {
    const int col = (j * kNormThreads + threadIdx.x) * 8;
    if (col < hidden) {
      const uint32_t ww[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
      uint32_t o[4], ro[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = pack_bf16x2(bf16_lo(ww[e]) * (v[j][2 * e] * rs), bf16_hi(ww[e]) * (v[j][2 * e + 1] * rs));
        ro[e] = pack_bf16x2(v[j][2 * e], v[j][2 * e + 1]);
      }
      *reinterpret_cast<uint4*>(out + row * out_stride + col) = make_uint4(o[0], o[1], o[2], o[3]);
      if (residual != nullptr && residual_out != nullptr)
        *reinterpret_cast<uint4*>(residual_out + row * res_out_stride + col) = make_uint4(ro[0], ro[1], ro[2], ro[3]);
    }
  }
}

// ---------------------------------------------------------------- SiLU * mul ------------

constexpr int kActThreads = 256;

// out[r, c] = bf16(silu(x[r, c]) * x[r, inter + c]) in fp32, c < inter; 8 columns per thread.
__global__ __launch_bounds__(kActThreads) void silu_and_mul_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, int32_t rows, int32_t inter,
    uint16_t* __restrict__ out, int64_t out_stride) {
  const int32_t vecs = inter / 8;
  const int64_t total = (int64_t)rows * vecs;
  for (int64_t i = (int64_t)blockIdx.x * kActThreads + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * kActThreads) {
    const int64_t r = i / vecs;
    const int32_t c = (int32_t)(i - r * vecs) * 8;
    const uint4 g = *reinterpret_cast<const uint4*>(x + r * x_stride + c);
    const uint4 u = *reinterpret_cast<const uint4*>(x + r * x_stride + inter + c);
    const uint32_t gg[4] = {g.x, g.y, g.z, g.w}, uu[4] = {u.x, u.y, u.z, u.w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float g0 = bf16_lo(gg[e]), g1 = bf16_hi(gg[e]);
      const float s0 = g0 / (1.0f + expf(-g0)), s1 = g1 / (1.0f + expf(-g1));
      o[e] = pack_bf16x2(s0 * bf16_lo(uu[e]), s1 * bf16_hi(uu[e]));
    }
    *reinterpret_cast<uint4*>(out + r * out_stride + c) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// ---------------------------------------------------------------- greedy LM head --------
//
// D = W_tile (vocab x K) . X^T (K x rows) on v_mfma_f32_32x32x16_bf16. A work-group owns 128
// vocabulary rows (32 per wavefront) and 32 * RT hidden rows; K is walked in chunks of 128.
// Each lane streams its vocabulary row from HBM with contiguous 16-byte loads: in k-step s of
// a chunk, MFMA k-slot (half h, element e) carries k = chunk + 64 h + 8 s + e. The B operand
// (the hidden rows, shared by every work-group and so L2-resident) is staged per chunk in LDS
// with the same k order, rows padded by 16 bytes so the 16-byte reads are conflict-free.
// The per-row best (bf16-rounded logit, lowest index on ties) is packed into one 64-bit key
// -- orderable logit bits above the complemented index -- and merged with a global atomic
// max; a finishing kernel turns keys into token ids.

constexpr int kLmThreads = 256;
constexpr int kLmVocabTile = 128;       // 4 wavefronts x 32 vocabulary rows
constexpr int kLmKChunk = 128;
constexpr int kLmLdsRow = kLmKChunk + 8;  // bf16 elements per staged row (16-byte pad)

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;

__device__ __forceinline__ uint64_t logit_key(float v, uint32_t idx) {
  const uint32_t b = __float_as_uint(v);
  const uint32_t ord = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return ((uint64_t)ord << 32) | (uint64_t)(~idx);
}

template <int RT>
__global__ __launch_bounds__(kLmThreads, 2) void lm_head_greedy_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const int32_t* __restrict__ cu_rows,
    const uint16_t* __restrict__ w, int64_t w_stride, int32_t rows, int32_t vocab, int32_t k_dim,
    unsigned long long* __restrict__ keys) {
  constexpr int MT = 32 * RT;
  __shared__ __attribute__((aligned(16))) uint16_t xs[MT * kLmLdsRow];
  __shared__ unsigned long long best_s[4][MT];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.y * MT;
  const int v_row = blockIdx.x * kLmVocabTile + wave * 32 + r;
  const uint16_t* wrow = w + (int64_t)(v_row < vocab ? v_row : vocab - 1) * w_stride + 64 * h;

  f32x16 acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;

  uint4 a_cur[8], a_nxt[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) a_cur[s] = *reinterpret_cast<const uint4*>(wrow + 8 * s);

  for (int kc = 0; kc < k_dim; kc += kLmKChunk) {
    const bool more = kc + kLmKChunk < k_dim;
    if (more) {
#pragma unroll
      for (int s = 0; s < 8; ++s)
        a_nxt[s] = *reinterpret_cast<const uint4*>(wrow + kc + kLmKChunk + 8 * s);
    }
    // stage the chunk of the hidden rows: MT rows x 16 pieces of 16 bytes
    __syncthreads();  // the previous chunk's reads are done
#pragma unroll
    for (int p = threadIdx.x; p < MT * 16; p += kLmThreads) {
      const int row = p >> 4, piece = p & 15;
      const int m = m0 + row;
      uint4 val = make_uint4(0, 0, 0, 0);
      if (m < rows) {
        // last row of sequence m when selecting (llm_head.py:61-63); a padded sequence
        // (zeroed cu_seqlens tail) has no row and contributes zeros
        const int src = cu_rows != nullptr ? cu_rows[m + 1] - 1 : m;
        if (src >= 0)
          val = *reinterpret_cast<const uint4*>(x + (int64_t)src * x_stride + kc + piece * 8);
      }
      *reinterpret_cast<uint4*>(xs + row * kLmLdsRow + piece * 8) = val;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const bf16x8_t av = __builtin_bit_cast(bf16x8_t, a_cur[s]);
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const uint4 bw = *reinterpret_cast<const uint4*>(xs + (32 * t + r) * kLmLdsRow + 64 * h + 8 * s);
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8_t, bw), acc[t], 0, 0, 0);
      }
    }
    if (more) {
#pragma unroll
      for (int s = 0; s < 8; ++s) a_cur[s] = a_nxt[s];
    }
  }

  // D layout: lane holds column (hidden row) 32 t + r and vocab rows 8 (i >> 2) + 4 h + (i & 3)
  const int v_base = blockIdx.x * kLmVocabTile + wave * 32;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    unsigned long long best = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int v = v_base + 8 * (i >> 2) + 4 * h + (i & 3);
      if (v < vocab) {
        const unsigned long long key = logit_key(round_to_bf16(acc[t][i]), (uint32_t)v);
        best = key > best ? key : best;
      }
    }
    const unsigned long long other = __shfl_xor(best, 32, kWave);
    best = other > best ? other : best;
    if (h == 0) best_s[wave][32 * t + r] = best;
  }
  __syncthreads();
  for (int j = threadIdx.x; j < MT; j += kLmThreads) {
    unsigned long long b = best_s[0][j];
#pragma unroll
    for (int q = 1; q < 4; ++q) b = best_s[q][j] > b ? best_s[q][j] : b;
    if (m0 + j < rows) atomicMax(keys + m0 + j, b);
  }
}

// Resident variant for hidden <= kLmResidentMaxK: a persistent work-group (one per CU) keeps
// its group of up to 64 hidden rows in LDS for the whole call and walks vocabulary tiles,
// so the hidden rows cross from L2 once per work-group instead of once per tile. The
// `groups` work-groups that cover the row groups of one vocabulary sequence have linear
// ids l, l + 8, ... and so sit on one XCD: each weight tile comes from HBM once and is
// shared through that XCD's L2.
constexpr int kLmResidentMaxK = 1024;
constexpr int kLmResidentRows = 64;
constexpr int kLmResidentWaves = 8;
constexpr int kLmResidentThreads = kLmResidentWaves * 64;
constexpr int kLmResidentTile = kLmResidentWaves * 32;  // vocabulary rows per tile

template <int RT>
__global__ __launch_bounds__(kLmResidentThreads, 1) void lm_head_resident_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const int32_t* __restrict__ cu_rows,
    const uint16_t* __restrict__ w, int64_t w_stride, int32_t rows, int32_t vocab, int32_t k_dim,
    int32_t groups, unsigned long long* __restrict__ keys) {
  constexpr int MT = 32 * RT;
  constexpr int kRowElems = kLmResidentMaxK + 8;  // staged row with a 16-byte pad
  __shared__ __attribute__((aligned(16))) uint16_t xs[MT * kRowElems];
  __shared__ unsigned long long best_s[kLmResidentWaves][MT];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r = lane & 31, h = lane >> 5;
  const int j = blockIdx.x >> 3;
  const int rg = j % groups;                          // row group
  const int rank = (j / groups) * 8 + (blockIdx.x & 7);  // position in the vocabulary walk
  const int nrank = gridDim.x / groups;
  const int m0 = rg * MT;

  // stage the group's hidden rows (the last row of sequence m when selecting,
  // llm_head.py:61-63; padded sequences and rows past `rows` stage zeros)
  const int pieces = k_dim / 8;
  for (int p = threadIdx.x; p < MT * pieces; p += kLmResidentThreads) {
    const int row = p / pieces, piece = p - row * pieces;
    const int m = m0 + row;
    uint4 val = make_uint4(0, 0, 0, 0);
    if (m < rows) {
      const int src = cu_rows != nullptr ? cu_rows[m + 1] - 1 : m;
      if (src >= 0) val = *reinterpret_cast<const uint4*>(x + (int64_t)src * x_stride + piece * 8);
    }
    *reinterpret_cast<uint4*>(xs + row * kRowElems + piece * 8) = val;
  }
  __syncthreads();

  unsigned long long best[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) best[t] = 0;
  // One stream of (tile, chunk) steps: the weight chunk of step n + 2 is in flight while
  // step n runs, across tile boundaries too.
  const int ntiles = (vocab + kLmResidentTile - 1) / kLmResidentTile;
  const int nchunks = k_dim / kLmKChunk;
  const int my_tiles = rank < ntiles ? (ntiles - rank + nrank - 1) / nrank : 0;
  const int steps = my_tiles * nchunks;
  auto wchunk = [&](int step) {
    const int t = step / nchunks;
    const int c = step - t * nchunks;
    const int v_row = (rank + t * nrank) * kLmResidentTile + wave * 32 + r;
    return w + (int64_t)(v_row < vocab ? v_row : vocab - 1) * w_stride + 64 * h + c * kLmKChunk;
  };
  f32x16 acc[RT];
  auto run_step = [&](const uint4 (&a)[8], int step) {
    const int t = step / nchunks;
    const int c = step - t * nchunks;
    if (c == 0) {
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[q][i] = 0.f;
    }
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) {
      const bf16x8_t av = __builtin_bit_cast(bf16x8_t, a[s8]);
#pragma unroll
      for (int q = 0; q < RT; ++q) {
        const uint4 bw = *reinterpret_cast<const uint4*>(xs + (32 * q + r) * kRowElems + c * kLmKChunk + 64 * h + 8 * s8);
        acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8_t, bw), acc[q], 0, 0, 0);
      }
    }
    if (c == nchunks - 1) {
      // D layout: lane holds column (hidden row) 32 q + r and vocab rows 8 (i >> 2) + 4 h + (i & 3)
      const int v_base = (rank + t * nrank) * kLmResidentTile + wave * 32;
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int v = v_base + 8 * (i >> 2) + 4 * h + (i & 3);
          if (v < vocab) {
            const unsigned long long key = logit_key(round_to_bf16(acc[q][i]), (uint32_t)v);
            best[q] = key > best[q] ? key : best[q];
          }
        }
    }
  };
  uint4 a0[8], a1[8];
  if (steps > 0) {
    const uint16_t* p0 = wchunk(0);
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) a0[s8] = *reinterpret_cast<const uint4*>(p0 + 8 * s8);
  }
  if (steps > 1) {
    const uint16_t* p1 = wchunk(1);
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) a1[s8] = *reinterpret_cast<const uint4*>(p1 + 8 * s8);
  }
  for (int step = 0; step < steps; step += 2) {
    run_step(a0, step);
    if (step + 2 < steps) {
      const uint16_t* pn = wchunk(step + 2);
#pragma unroll
      for (int s8 = 0; s8 < 8; ++s8) a0[s8] = *reinterpret_cast<const uint4*>(pn + 8 * s8);
    }
    if (step + 1 >= steps) break;
    run_step(a1, step + 1);
    if (step + 3 < steps) {
      const uint16_t* pn = wchunk(step + 3);
#pragma unroll
      for (int s8 = 0; s8 < 8; ++s8) a1[s8] = *reinterpret_cast<const uint4*>(pn + 8 * s8);
    }
  }
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const unsigned long long other = __shfl_xor(best[t], 32, kWave);
    const unsigned long long b = other > best[t] ? other : best[t];
    if (h == 0) best_s[wave][32 * t + r] = b;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < MT; q += kLmResidentThreads) {
    unsigned long long b = best_s[0][q];
#pragma unroll
    for (int wv = 1; wv < kLmResidentWaves; ++wv) b = best_s[wv][q] > b ? best_s[wv][q] : b;
    if (m0 + q < rows) atomicMax(keys + m0 + q, b);
  }
}

// Variant for up to 64 hidden rows of kLmSplitHidden columns: a persistent work-group per CU walks
// 32-row vocabulary tiles, and its eight wavefronts split K: wavefront w multiplies columns
// [128 w, 128 w + 128) of the tile by those of the hidden rows, which it holds in registers for the
// whole call (32 RT of them). A wavefront's slice of a tile (32 rows x 256 bytes) goes from memory to
// its own 8 KiB of LDS without registers, four full rows' pieces per instruction, one tile ahead and
// without a barrier; the eight partial sums of a tile meet in the same LDS.
//
// What bounds lm_head_resident_kernel: every lane loads its own vocabulary row, so each load
// instruction touches 64 cache lines, 16 bytes of each, at the L1's tag rate. Whole call over 151936
// vocabulary rows, us, that kernel -> this one: 1 row 62.0 -> 54.5, 32 64.3 -> 61.5, 64 68.7 -> 63.8.
// What is left: the wavefronts' MFMAs and sums alternate behind barriers. Which calls take it:
// lm_split_pays.
constexpr int kLmSplitWaves = 8;
constexpr int kLmSplitHidden = kLmSplitWaves * kLmKChunk;  // 1024: every wavefront has a K slice
constexpr int kLmSplitThreads = kLmSplitWaves * 64;
constexpr int kLmSplitRows = 128;       // hidden rows per work-group
constexpr int kLmSplitTile = 32;        // vocabulary rows per tile
constexpr int kLmSliceBytes = 32 * 256;  // a wavefront's slice of 32 rows
constexpr int kLmStageBytes = kLmSplitWaves * kLmSliceBytes;

typedef __attribute__((address_space(3))) char lds_char;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// 16 bytes per lane from base + off to LDS offset lds + 16 lane.
__device__ __forceinline__ void lm_load16(uint64_t base, uint32_t off, int lds) {
  const uint64_t b = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)base) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(base >> 32)) << 32;
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(off), "s"(b)
      : "m0", "memory");
}
// Waits until at most N vector memory operations of this wavefront are in flight.
template <int N>
__device__ __forceinline__ void lm_wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// LDS-only barrier (the next tile's loads stay in flight).
__device__ __forceinline__ void lm_barrier() {
  __builtin_amdgcn_s_waitcnt((15 & 15) | ((63 >> 4) << 14) | (7 << 4) | (0 << 8));
  asm volatile("s_barrier" ::: "memory");
}

template <int RT>
__global__ __launch_bounds__(kLmSplitThreads, 2) void lm_head_split_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const int32_t* __restrict__ cu_rows,
    const uint16_t* __restrict__ w, int64_t w_stride, int32_t rows, int32_t vocab,
    unsigned long long* __restrict__ keys) {
  static_assert(RT <= 2, "two row blocks of partial sums fill a slice");
  __shared__ __attribute__((aligned(1024))) char smem_[2 * kLmStageBytes];
  lds_char* const smem = (lds_char*)smem_;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r = lane & 31, h = lane >> 5;
  const int rank = blockIdx.x;
  const int nrank = gridDim.x;
  const int slice0 = (int)(uintptr_t)smem + wave * kLmSliceBytes;  // this wavefront's slice, stage 0
  lds_char* const own = smem + wave * kLmSliceBytes;
  // load i of a slice: rows 4 i + (lane >> 4), 16-byte chunk c of row n in slot c ^ (n & 15)
  const int lrow = lane >> 4;
  const int lchunk = (lane & 15) ^ lrow;  // of load 0; load i: ^ 4 (i & 3)
  // MFMA operand of K step s8: row r, chunk 2 s8 + h
  const int rofs = r * 256;
  const auto read = [&](int stage, int s8) {
    return *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(
        own + stage * kLmStageBytes + rofs + (((2 * s8 + h) ^ (r & 15)) << 4));
  };

  // the hidden rows' slices through LDS (the last row of sequence m when selecting,
  // llm_head.py:61-63; padded sequences and rows past `rows` are zero)
  u32x4_t xr[RT][8];
  const auto src_row = [&](int m) { return m >= rows ? -1 : cu_rows != nullptr ? cu_rows[m + 1] - 1 : m; };
  const auto load_x = [&](int q) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int src = src_row(32 * q + 4 * i + lrow);
      if (src >= 0) {
        const uint16_t* p = x + (int64_t)src * x_stride + wave * kLmKChunk + (lchunk ^ (4 * (i & 3))) * 8;
        asm volatile(
            "s_mov_b32 m0, %0\n\t"
            "s_nop 0\n\t"
            "global_load_lds_dwordx4 %1, off"
            :
            : "s"(__builtin_amdgcn_readfirstlane(slice0 + q * kLmStageBytes + 1024 * i)), "v"(p)
            : "m0", "memory");
      }
    }
  };
  const auto take_x = [&](int q) {
    const bool live = src_row(32 * q + r) >= 0;
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) {
      const u32x4_t v = read(q, s8);
      xr[q][s8] = live ? v : u32x4_t{0, 0, 0, 0};
    }
  };
#pragma unroll
  for (int q = 0; q < RT; ++q) load_x(q);
  lm_wait_vm<0>();
#pragma unroll
  for (int q = 0; q < RT; ++q) {
    take_x(q);
    asm volatile("" : "+v"(xr[q][0]), "+v"(xr[q][1]), "+v"(xr[q][2]), "+v"(xr[q][3]), "+v"(xr[q][4]),
                 "+v"(xr[q][5]), "+v"(xr[q][6]), "+v"(xr[q][7]));  // read before the stage is loaded again
  }

  const int ntiles = (vocab + kLmSplitTile - 1) / kLmSplitTile;
  const auto load_tile = [&](int t, int stage) {
    if (t >= ntiles) return;
    const uint64_t base = (uint64_t)(w + (int64_t)t * kLmSplitTile * w_stride + wave * kLmKChunk);
    const int last = vocab - 1 - t * kLmSplitTile;  // rows past the vocabulary re-read the last one
#pragma unroll
    for (int i = 0; i < 8; ++i)
      lm_load16(base, (uint32_t)(min(4 * i + lrow, last) * (int)w_stride + (lchunk ^ (4 * (i & 3))) * 8) * 2,
                slice0 + stage * kLmStageBytes + 1024 * i);
  };
  unsigned long long best = 0;
  load_tile(rank, 0);
  load_tile(rank + nrank, 1);
  int stage = 0;
  for (int t = rank; t < ntiles; t += nrank, stage ^= 1) {
    f32x16 acc[RT];
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[q][i] = 0.f;
    if (t + nrank < ntiles)
      lm_wait_vm<8>();
    else
      lm_wait_vm<0>();
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) {
      const bf16x8_t av = __builtin_bit_cast(bf16x8_t, read(stage, s8));
#pragma unroll
      for (int q = 0; q < RT; ++q)
        acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8_t, xr[q][s8]), acc[q], 0, 0, 0);
    }
    // D layout: lane holds hidden row 32 q + r and vocabulary rows 8 (i >> 2) + 4 h + (i & 3).
    // Wavefront v sums quad v & 3 of row block v >> 2 over the slices, in K order.
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<__attribute__((address_space(3))) f32x4_t*>(own + stage * kLmStageBytes + (4 * q + i) * 1024 +
                                                                     lane * 16) =
            f32x4_t{acc[q][4 * i], acc[q][4 * i + 1], acc[q][4 * i + 2], acc[q][4 * i + 3]};
    lm_barrier();
    if ((wave >> 2) < RT) {
      const lds_char* const part = smem + stage * kLmStageBytes + wave * 1024 + lane * 16;
      f32x4_t sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u0 = 0; u0 < kLmSplitWaves; u0 += 4) {
        f32x4_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          v[u] = *reinterpret_cast<const __attribute__((address_space(3))) f32x4_t*>(part + (u0 + u) * kLmSliceBytes);
#pragma unroll
        for (int u = 0; u < 4; ++u) sum += v[u];
      }
      const int vrow = t * kLmSplitTile + 8 * (wave & 3) + 4 * h;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (vrow + e < vocab) {
          const unsigned long long key = logit_key(round_to_bf16(sum[e]), (uint32_t)(vrow + e));
          best = key > best ? key : best;
        }
    }
    lm_barrier();
    load_tile(t + 2 * nrank, stage);
  }
  // the best of a hidden row over its quads (wavefronts) and lane halves
  const unsigned long long other = __shfl_xor(best, 32, kWave);
  const unsigned long long b = other > best ? other : best;
  const int m = 32 * (wave >> 2) + r;
  if (h == 0 && (wave >> 2) < RT && m < rows && b != 0) atomicMax(keys + m, b);
}

// The same with four K slices of 256 columns and two halves of 128 hidden rows: wavefront k + 4 m
// multiplies slice k by row blocks 2 m and 2 m + 1, so half as many partial sums meet; the two
// wavefronts of a slice share it (and load half of its rows each). It takes more than kLmSplit4Rows
// hidden rows (below, a second half would hold no rows) of a hidden size that its slices divide; with
// three slices a quarter of the wavefronts idles. Whole call over 151936 vocabulary rows, us,
// lm_head_resident_kernel -> this one: 96 rows 92.5 -> 80.7, 128 rows 94.3 -> 81.1, 129 rows 131.5 ->
// 116.9, 512 rows 290.0 -> 218.6.
constexpr int kLmSplit4Rows = 64;

__global__ __launch_bounds__(kLmSplitThreads, 2) void lm_head_split4_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const int32_t* __restrict__ cu_rows,
    const uint16_t* __restrict__ w, int64_t w_stride, int32_t rows, int32_t vocab, int32_t k_dim,
    int32_t groups, unsigned long long* __restrict__ keys) {
  constexpr int kCols = 256;
  constexpr int kSlice = 32 * kCols * 2;  // 32 rows x 512 bytes
  __shared__ __attribute__((aligned(1024))) char smem_[2 * kLmStageBytes];
  lds_char* const smem = (lds_char*)smem_;
  const int lds0 = (int)(uintptr_t)smem;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int ks = wave & 3, half_m = wave >> 2;
  const int r = lane & 31, h = lane >> 5;
  // the `groups` work-groups of one place in the vocabulary walk (row groups of 128) have linear
  // ids l, l + 8, ... and so share an XCD's L2
  const int j = blockIdx.x >> 3;
  const int rg = j % groups;
  const int rank = (j / groups) * 8 + (blockIdx.x & 7);
  const int nrank = gridDim.x / groups;
  const int m0 = rg * kLmSplitRows;
  const int nk = k_dim / kCols;
  const bool on = ks < nk;
  // 16-byte chunk c of row n of a slice in slot c ^ (n & 15); a load moves two rows
  const auto read = [&](const lds_char* slice, int s) {
    return *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(slice + r * (kCols * 2) +
                                                                            (((2 * s + h) ^ (r & 15)) << 4));
  };
  const auto src_row = [&](int m) { return m >= rows ? -1 : cu_rows != nullptr ? cu_rows[m + 1] - 1 : m; };

  // the hidden rows' slices, a block of 32 at a time through 16 KiB of the wavefront's own
  u32x4_t xr[2][16];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int mb = m0 + 32 * (2 * half_m + q);
    if (on) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = 2 * i + h;
        const int src = src_row(mb + row);
        if (src >= 0) {
          const uint16_t* p = x + (int64_t)src * x_stride + ks * kCols + (r ^ (row & 15)) * 8;
          asm volatile(
              "s_mov_b32 m0, %0\n\t"
              "s_nop 0\n\t"
              "global_load_lds_dwordx4 %1, off"
              :
              : "s"(__builtin_amdgcn_readfirstlane(lds0 + wave * kSlice + 1024 * i)), "v"(p)
              : "m0", "memory");
        }
      }
      lm_wait_vm<0>();
    }
    const bool live = on && src_row(mb + r) >= 0;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const u32x4_t v = read(smem + wave * kSlice, s);
      xr[q][s] = live ? v : u32x4_t{0, 0, 0, 0};
      asm volatile("" : "+v"(xr[q][s]));  // read before the next rows arrive
    }
  }
  lm_barrier();

  const int ntiles = (vocab + kLmSplitTile - 1) / kLmSplitTile;
  const auto load_tile = [&](int t, int stage) {
    if (!on || t >= ntiles) return;
    const uint64_t base = (uint64_t)(w + (int64_t)t * kLmSplitTile * w_stride + ks * kCols);
    const int last = vocab - 1 - t * kLmSplitTile;  // rows past the vocabulary re-read the last one
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 16 * half_m + 2 * i + h;
      lm_load16(base, (uint32_t)(min(row, last) * (int)w_stride + (r ^ (row & 15)) * 8) * 2,
                lds0 + stage * kLmStageBytes + ks * kSlice + (8 * half_m + i) * 1024);
    }
  };
  unsigned long long best[2] = {0, 0};
  load_tile(rank, 0);
  load_tile(rank + nrank, 1);
  int stage = 0;
  for (int t = rank; t < ntiles; t += nrank, stage ^= 1) {
    lds_char* const st = smem + stage * kLmStageBytes;
    f32x16 acc[2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[q][i] = 0.f;
    if (t + nrank < ntiles)
      lm_wait_vm<8>();
    else
      lm_wait_vm<0>();
    lm_barrier();  // both halves of the slices have landed
    if (on) {
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const bf16x8_t av = __builtin_bit_cast(bf16x8_t, read(st + ks * kSlice, s));
#pragma unroll
        for (int q = 0; q < 2; ++q)
          acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, __builtin_bit_cast(bf16x8_t, xr[q][s]), acc[q], 0, 0, 0);
      }
    }
    lm_barrier();  // the slices have been read: partial sums take their place
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<__attribute__((address_space(3))) f32x4_t*>(st + wave * kLmSliceBytes + (4 * q + i) * 1024 +
                                                                     lane * 16) =
            f32x4_t{acc[q][4 * i], acc[q][4 * i + 1], acc[q][4 * i + 2], acc[q][4 * i + 3]};
    lm_barrier();
    // wavefront v sums quad v & 3 of row blocks v >> 2 and 2 + (v >> 2) over the slices, in K order
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int blk = 2 * p + (wave >> 2);
      const lds_char* const part = st + (blk >> 1) * 4 * kLmSliceBytes + (4 * (blk & 1) + (wave & 3)) * 1024 + lane * 16;
      f32x4_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        v[u] = *reinterpret_cast<const __attribute__((address_space(3))) f32x4_t*>(part + u * kLmSliceBytes);
      const f32x4_t sum = ((v[0] + v[1]) + v[2]) + v[3];  // slices past hidden are zero
      const int vrow = t * kLmSplitTile + 8 * (wave & 3) + 4 * h;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (vrow + e < vocab) {
          const unsigned long long key = logit_key(round_to_bf16(sum[e]), (uint32_t)(vrow + e));
          best[p] = key > best[p] ? key : best[p];
        }
    }
    lm_barrier();
    load_tile(t + 2 * nrank, stage);
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const unsigned long long other = __shfl_xor(best[p], 32, kWave);
    const unsigned long long b = other > best[p] ? other : best[p];
    const int m = m0 + 32 * (2 * p + (wave >> 2)) + r;
    if (h == 0 && m < rows && b != 0) atomicMax(keys + m, b);
  }
}

__global__ void lm_keys_clear_kernel(unsigned long long* keys, int32_t rows) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < rows) keys[i] = 0ull;
}

__global__ void lm_keys_to_ids_kernel(const unsigned long long* keys, int32_t rows, int32_t* ids) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < rows) ids[i] = (int32_t)(~(uint32_t)(keys[i] & 0xffffffffull));
}

}  // namespace

hipError_t launch_add_rmsnorm(const void* x, int64_t x_stride, const void* residual,
                              int64_t res_stride, const void* weight, float eps, int32_t rows,
                              int32_t hidden, void* out, int64_t out_stride, void* residual_out,
                              int64_t res_out_stride, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const int vecs = (hidden / 8 + kNormThreads - 1) / kNormThreads;
  auto* xp = static_cast<const uint16_t*>(x);
  auto* rp = static_cast<const uint16_t*>(residual);
  auto* wp = static_cast<const uint16_t*>(weight);
  auto* op = static_cast<uint16_t*>(out);
  auto* rop = static_cast<uint16_t*>(residual_out);
  switch (vecs) {
    case 1: hipLaunchKernelGGL(add_rmsnorm_kernel<1>, dim3(rows), dim3(kNormThreads), 0, stream, xp, x_stride, rp, res_stride, wp, eps, hidden, op, out_stride, rop, res_out_stride); break;
    case 2: hipLaunchKernelGGL(add_rmsnorm_kernel<2>, dim3(rows), dim3(kNormThreads), 0, stream, xp, x_stride, rp, res_stride, wp, eps, hidden, op, out_stride, rop, res_out_stride); break;
    case 3: hipLaunchKernelGGL(add_rmsnorm_kernel<3>, dim3(rows), dim3(kNormThreads), 0, stream, xp, x_stride, rp, res_stride, wp, eps, hidden, op, out_stride, rop, res_out_stride); break;
    case 4: hipLaunchKernelGGL(add_rmsnorm_kernel<4>, dim3(rows), dim3(kNormThreads), 0, stream, xp, x_stride, rp, res_stride, wp, eps, hidden, op, out_stride, rop, res_out_stride); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_silu_and_mul(const void* x, int64_t x_stride, int32_t rows, int32_t inter,
                               void* out, int64_t out_stride, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const int64_t total = (int64_t)rows * (inter / 8);
  int64_t blocks = (total + kActThreads - 1) / kActThreads;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(silu_and_mul_kernel, dim3((unsigned)blocks), dim3(kActThreads), 0, stream,
                     static_cast<const uint16_t*>(x), x_stride, rows, inter,
                     static_cast<uint16_t*>(out), out_stride);
  return hipGetLastError();
}

// Whether the split kernels are the faster ones. A persistent work-group pays its start (the hidden
// rows into registers, two tiles on their way) once for the tiles it walks, and a K slice without
// columns is a wavefront without work. lm_head_resident_kernel / split kernels, time ratio by tiles per work-group (2.3, 4.6, 9.3, 18.5):
//   hidden 1024, 1-64 rows     0.84-1.15  0.77-0.90  0.99-1.13  1.05-1.14
//   hidden 1024, 65-128 rows   0.80-0.83  1.03-1.05  1.06-1.08  1.14-1.16
//   hidden 1024, more rows     1.03-1.05  0.97-1.42  1.02-1.58  1.10-1.46
//   hidden 768, 129-192 rows   0.87       0.81       0.85       0.90-0.94
//   hidden 768, more rows      0.88-0.93  1.08-1.32  1.06-1.30  1.01-1.21
// hidden 768 with fewer rows 0.67-1.02, hidden 512 0.53-0.92 and 128 0.30-0.69 (896: 0.71-1.20, not a
// multiple of 256).
bool lm_split_pays(int32_t rows, int32_t vocab, int32_t k_dim, int32_t groups, int32_t cus) {
  const int64_t tiles = (int64_t)((vocab + kLmSplitTile - 1) / kLmSplitTile) * groups;
  if (k_dim == kLmSplitHidden) return tiles >= (int64_t)cus * (rows <= kLmSplit4Rows ? 8 : rows <= kLmSplitRows ? 4 : 2);
  return k_dim == kLmSplitHidden * 3 / 4 && rows > 3 * kLmSplitRows / 2 && tiles >= 4 * (int64_t)cus;
}

hipError_t launch_lm_head_greedy(const void* x, int64_t x_stride, const int32_t* cu_rows,
                                 const void* w, int64_t w_stride, int32_t rows, int32_t vocab,
                                 int32_t k_dim, unsigned long long* keys, int32_t* ids,
                                 hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const unsigned small = (unsigned)((rows + 255) / 256);
  hipLaunchKernelGGL(lm_keys_clear_kernel, dim3(small), dim3(256), 0, stream, keys, rows);
  const unsigned vt = (unsigned)((vocab + kLmVocabTile - 1) / kLmVocabTile);
  auto* xp = static_cast<const uint16_t*>(x);
  auto* wp = static_cast<const uint16_t*>(w);
  static int cus_cached = 0;
  if (cus_cached == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
    cus_cached = cus;
  }
  // a persistent grid of whole XCD rounds of every row group
  const auto grid_of = [](int groups) { return std::max(cus_cached / (8 * groups), 1) * 8 * groups; };
  const int split_groups = (rows + kLmSplitRows - 1) / kLmSplitRows;
  // (a split tile's offsets fit 32 bits)
  if (w_stride < (1 << 25) && lm_split_pays(rows, vocab, k_dim, split_groups, cus_cached)) {
    const dim3 grid(grid_of(split_groups));
    if (rows > kLmSplit4Rows)
      hipLaunchKernelGGL(lm_head_split4_kernel, grid, dim3(kLmSplitThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, k_dim, split_groups, keys);
    else if (rows > 32)
      hipLaunchKernelGGL(lm_head_split_kernel<2>, grid, dim3(kLmSplitThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, keys);
    else
      hipLaunchKernelGGL(lm_head_split_kernel<1>, grid, dim3(kLmSplitThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, keys);
  } else if (k_dim <= kLmResidentMaxK) {
    const int groups = (rows + kLmResidentRows - 1) / kLmResidentRows;
    const dim3 grid(grid_of(groups));
    if (rows <= 32)
      hipLaunchKernelGGL(lm_head_resident_kernel<1>, grid, dim3(kLmResidentThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, k_dim, groups, keys);
    else
      hipLaunchKernelGGL(lm_head_resident_kernel<2>, grid, dim3(kLmResidentThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, k_dim, groups, keys);
  } else if (rows <= 32) {
    hipLaunchKernelGGL(lm_head_greedy_kernel<1>, dim3(vt, 1), dim3(kLmThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, k_dim, keys);
  } else if (rows <= 64) {
    hipLaunchKernelGGL(lm_head_greedy_kernel<2>, dim3(vt, 1), dim3(kLmThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, k_dim, keys);
  } else {
    hipLaunchKernelGGL(lm_head_greedy_kernel<4>, dim3(vt, (unsigned)((rows + 127) / 128)), dim3(kLmThreads), 0, stream, xp, x_stride, cu_rows, wp, w_stride, rows, vocab, k_dim, keys);
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(lm_keys_to_ids_kernel, dim3(small), dim3(256), 0, stream, keys, rows, ids);
  return hipGetLastError();
}

}  // namespace pk
