// Chunked-prefill / dense varlen attention on bf16 MFMA for gfx950.
//
// Reference semantics: flash_attn_varlen_func(..., causal=True, block_table) at
// src/layers/attention.py:95-104 for sequences with Lq > 1 query rows. Row i of a
// sequence with Lq rows and Lk keys sees keys t <= i + (Lk - Lq) (bottom-right
// alignment, the cached prefix P = Lk - Lq precedes the chunk; model_runner.py:186-190).
// Keys come through the block table (paged, chunked prefill / prefix-cache hits) or
// from fresh rows at cu_seqlens_k (flat, all-fresh prompts).
//
// Work unit: 256 query rows = TM = 256 / G query tokens x the G query heads of one kv
// head g, so each K/V tile staged in LDS serves the whole GQA group. Two kernels own units, one
// work-group per CU: prefill_kernel with four wavefronts (one per SIMD, the whole register file) of
// two blocks of 32 rows, and prefill_w8_kernel, for small calls, with eight of one block; a block is
// 32 consecutive tokens of one head (TM >= 32 for every GQA group built).
//
// Three launches, all sized on the host without reading device memory:
//   1. plan (one work-group): reads cu_seqlens_q/k, counts each unit's key tiles under
//      its causal limit, picks a split size T = max(8, kSplitNum / kSplitDen x total tiles
//      / pool) tiles and writes the work list: every unit longer than T is cut into equal
//      key ranges. Long items come first (eight length buckets, four for small calls).
//   2. prefill (a persistent pool of one work-group per CU): each work-group starts on the item
//      of its own index, then claims items from the sub-queue of its XCD (item i belongs to
//      sub-queue i mod 8, which for 8 kv heads is kv head i mod 8, so a head's K/V stays in one
//      XCD's L2), then steals from the other sub-queues. An unsplit item writes bf16 rows; a
//      split item writes its own output in bf16 and (max, sum) per row.
//   3. merge: combines the partials of every split unit, then the decode rows' partials
//      left by the call's decode launch (paged_decode.hip), which needs no combine launch.
// The split bounds the longest chain of dependent tiles (a long cached prefix would
// otherwise keep one work-group busy long after the rest of the GPU has finished).
//
// prefill_kernel, per step of 32 keys (half a tile), per wavefront and 32-row block:
//   S^T (32 keys x 32 rows) = K (32 x 128) . Q^T (128 x 32)    8 v_mfma_f32_32x32x16_bf16
//   P = 2^(S - reference of the row) (a lane owns one query row)
//   O^T (128 x 32)         += V^T (128 x 32) . P^T (32 x 32)   8 v_mfma_f32_32x32x16_bf16
// The three parts of consecutive steps run as one instruction stream (pf_iteration). K and V
// tiles go from memory to LDS without registers (global_load_lds), K four tiles and V three tiles
// deep. The P.V A operand comes from the LDS transpose read. P^T never leaves registers: the
// S^T accumulator layout already holds, per lane, the keys the P.V B operand needs once
// the k-order of the instruction is permuted (same permutation on the V side).
#include <algorithm>

#include "decode_core.h"

namespace pk {
namespace {

constexpr int kTileKeys = 64;          // keys per K/V tile
#ifndef PK_PREFILL_ROW_BLOCKS
#define PK_PREFILL_ROW_BLOCKS 1
#endif
// A wavefront owns kRowBlocks blocks of 32 query rows; every K and V operand it reads from
// LDS serves all of its blocks, so LDS read traffic per flop falls as 1 / kRowBlocks.
constexpr int kRowBlocks = PK_PREFILL_ROW_BLOCKS;
static_assert(kRowBlocks == 1 || kRowBlocks == 2, "row blocks per wavefront");
constexpr int kPrefillWaves = 8 / kRowBlocks;           // 256 rows per work-group
constexpr int kPrefillThreads = kPrefillWaves * 64;
constexpr int kWavesPerSimd = 2 / kRowBlocks;           // register file: 512 / this per lane
constexpr int kRowBytes = kHeadDim * 2;                  // one head's row of a K or V tile (256 B)
constexpr int kTileBytes = kTileKeys * kRowBytes;        // 16 KiB per operand per stage
constexpr int kPlanThreads = 1024;     // plan work-group
constexpr int kPlanCache = 2048;       // sequences whose lengths the plan keeps in LDS
constexpr int kMinSplitTiles = 8;      // never split a unit's keys below 512 per item
#ifndef PK_PREFILL_SPLIT_NUM
#define PK_PREFILL_SPLIT_NUM 2
#define PK_PREFILL_SPLIT_DEN 3
#endif
constexpr int kSplitNum = PK_PREFILL_SPLIT_NUM;  // split size = kSplitNum / kSplitDen x work per slot
constexpr int kSplitDen = PK_PREFILL_SPLIT_DEN;
constexpr int kMergeThreads = 256;     // merge: thread = row of the unit
constexpr int kMergeGroups = 1024;
constexpr int kMergeBatch = 8;         // merge: splits whose (max, sum) load in one batch
#ifndef PK_MERGE_LOADS
#define PK_MERGE_LOADS 4
#endif
constexpr int kMergeLoads = PK_MERGE_LOADS;  // merge: splits whose outputs load in one batch
#ifndef PK_PREFILL_BUCKETS
#define PK_PREFILL_BUCKETS 8
#endif
// Length buckets of the work list (longest first). prefill_kernel: 4 -> 8 took the dense prompts
// 144.4 -> 141.6 us and the long chunks 605 -> 594 us, 16 gave 146.3 and 594; prefill_w8_kernel
// keeps 4 (8: 31 prompts of 512 114.2 -> 118.9 us, 15 chunks of 100 over 4096 keys 117.5 -> 119.9).
constexpr int kLargeBuckets = PK_PREFILL_BUCKETS;
constexpr int kSmallBuckets = 4;
constexpr float kLazyLog2 = 8.f;       // reference max moves only when exceeded by 2^8

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;


// Value of lane l ^ 32 (the other half of the wavefront), one VALU swap.
__device__ __forceinline__ float swap_halves_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}
__device__ __forceinline__ float swap_halves_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  return __int_as_float(r[0]) + __int_as_float(r[1]);
}

// Work-group barrier for the LDS tiles: wait until this wavefront's LDS instructions have
// completed, then s_barrier. It is issued as an instruction of its own because
// __syncthreads() would also wait for every global load in flight (its fence waits for
// vmcnt(0)), including the next tile's loads that are meant to overlap the compute.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt((15 & 15) | ((63 >> 4) << 14) | (7 << 4) | (0 << 8));  // lgkmcnt(0) only
  asm volatile("s_barrier" ::: "memory");
}

// LDS tiles are stored unpadded, one 256-byte row per key, with the row's sixteen 16-byte
// chunks XOR-swizzled so that the MFMA operand reads hit distinct banks:
//   K: chunk c of row r lives in slot c ^ (r & 15)      (32 consecutive rows read chunk c)
//   V: chunk c of row r lives in slot c ^ ((2 r) & 15) ^ 8 (c & 2)
// A V transpose read serves 32 lanes per cycle: two 16-lane groups, each reading 4
// consecutive rows x 2 chunks, the second group the next two chunks. The XOR with 2 r
// spreads a group over 8 slots; the extra 8 (c & 2) puts the second group's chunks in the
// other 8 slots, so the 32 lanes hit all 64 banks once.
__device__ __forceinline__ int k_slot(int r, int c) { return c ^ (r & 15); }
__device__ __forceinline__ int v_slot(int r, int c) { return c ^ ((2 * r) & 15) ^ ((c & 2) << 2); }
// Inverse of v_slot: the chunk stored in slot s of row r (bit 1 of the chunk survives the
// first XOR, so it names the second one).
__device__ __forceinline__ int v_chunk(int r, int s) {
  const int y = s ^ ((2 * r) & 15);
  return y ^ ((y & 2) << 2);
}

// Keys [t0, t0 + 64) of kv head g move global -> registers -> LDS: wavefront w owns tile
// rows kRowsPerWave w .. kRowsPerWave (w + 1) - 1, four rows (1 KiB) per 16-byte load
// instruction, lane l carrying slot (l & 15) of row (l >> 4) and therefore the swizzled
// source chunk. The loads for tile n + 2 are issued before tile n is computed and written
// to LDS after tile n + 1 has been (register staging keeps them off the LDS while it
// serves the MFMA operands). Keys past Lk re-read the last key's row (same cache block,
// finite data); their scores are masked and their p is 0.
constexpr int kRowsPerWave = kTileKeys / kPrefillWaves;
constexpr int kLoadsPerOperand = kRowsPerWave / 4;


// Per-lane source byte offsets of the rows this lane moves.
struct LoadLanes {
  int k[kLoadsPerOperand];
  int v[kLoadsPerOperand];
};

__device__ __forceinline__ LoadLanes load_lanes(const AttnArgs& a, int wave, int lane, int last) {
  LoadLanes l;
  const int slot = lane & 15;
#pragma unroll
  for (int i = 0; i < kLoadsPerOperand; ++i) {
    const int r = kRowsPerWave * wave + 4 * i + (lane >> 4);  // tile row this lane fills
    const int rs = min(r, last);                              // source row (clamped on the last tile)
    l.k[i] = (rs * (int)a.k_row_stride + (slot ^ (r & 15)) * 8) * 2;
    l.v[i] = (rs * (int)a.v_row_stride + v_chunk(r, slot) * 8) * 2;
  }
  return l;
}

struct KvRegs {
  u32x4 k[kLoadsPerOperand];
  u32x4 v[kLoadsPerOperand];
};

// The lane's 16-byte loads of one tile from K and V rows starting at kbase / vbase. (Buffer
// loads over the tile's rows, which keep no 64-bit lane address, measured 2-4% slower on
// the prefill batches.)
__device__ __forceinline__ void load_rows(const uint16_t* kbase, const uint16_t* vbase, const LoadLanes& l,
                                          KvRegs& R) {
#pragma unroll
  for (int i = 0; i < kLoadsPerOperand; ++i) {
    R.k[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(kbase) + l.k[i]);
    R.v[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(vbase) + l.v[i]);
  }
}

template <bool PAGED>
__device__ __forceinline__ void load_tile_regs(const AttnArgs& a, int b, int k0, int Lk, int g, int bt_lane, int wave,
                                               int lane, int t0, const LoadLanes& full_lanes, KvRegs& R) {
  const uint16_t* kbase;
  const uint16_t* vbase;
  if constexpr (PAGED) {
    const int j = t0 / a.block_size;  // block_size % 64 == 0: the tile sits inside one block
    const int blk = j < kWave ? __builtin_amdgcn_readlane(bt_lane, j)
                              : __builtin_amdgcn_readfirstlane(a.block_table[(int64_t)b * a.bt_stride + j]);
    const int off = t0 % a.block_size;
    kbase = a.k + (int64_t)blk * a.k_block_stride + (int64_t)off * a.k_row_stride;
    vbase = a.v + (int64_t)blk * a.v_block_stride + (int64_t)off * a.v_row_stride;
  } else {
    kbase = a.k + (int64_t)(k0 + t0) * a.k_row_stride;
    vbase = a.v + (int64_t)(k0 + t0) * a.v_row_stride;
  }
  kbase += g * kHeadDim;
  vbase += g * kHeadDim;
  load_rows(kbase, vbase, (t0 + kTileKeys <= Lk) ? full_lanes : load_lanes(a, wave, lane, Lk - 1 - t0), R);
}

__device__ __forceinline__ void store_tile_lds(const KvRegs& R, lds_char* kdst, lds_char* vdst, int wave, int lane) {
#pragma unroll
  for (int i = 0; i < kLoadsPerOperand; ++i) {
    const int off = (kRowsPerWave * wave + 4 * i) * kRowBytes + lane * 16;
    *reinterpret_cast<__attribute__((address_space(3))) u32x4*>(kdst + off) = R.k[i];
    *reinterpret_cast<__attribute__((address_space(3))) u32x4*>(vdst + off) = R.v[i];
  }
}

// Online softmax of one 32-row block's S^T tile (64 keys) in place: scores become p, the
// row sums move on, and p is packed to bf16 as the P.V B operand. S^T element rr of
// half-tile mb is key t0 + 32 mb + 8 (rr >> 2) + 4 half + (rr & 3). Raw scores are
// compared (the scale is positive) and scaled inside the exponent's FMA.
// Lazy rescaling: exponentials are taken against a reference max m_i (exp2 domain) that
// moves only when some row's tile max exceeds it by more than kLazyLog2; then every row
// moves to its running max and the numerator and sum are rescaled. p <= 2^kLazyLog2, and
// numerator and sum share the reference, so o / l is unchanged.
// The parts of softmax_block over NB half-tiles of 32 keys (element rr of half-tile mb is
// key t0 + 32 mb + 8 (rr >> 2) + 4 half + (rr & 3)): the mask (diagonal tiles) and the
// row's max in the exp2 domain ...
template <int NB>
__device__ __forceinline__ void softmax_mask(f32x16 (&s)[NB], int t0, int lim, int half) {
#pragma unroll
  for (int mb = 0; mb < NB; ++mb)
#pragma unroll
    for (int rr = 0; rr < 16; ++rr)
      if (t0 + mb * 32 + 8 * (rr >> 2) + 4 * half + (rr & 3) > lim) s[mb][rr] = -INFINITY;
}

template <int NB, bool MASK>
__device__ __forceinline__ float softmax_max(f32x16 (&s)[NB], int t0, int lim, float scale_log2, int half) {
  if constexpr (MASK) softmax_mask<NB>(s, t0, lim, half);
  float tmax = -INFINITY;
#pragma unroll
  for (int mb = 0; mb < NB; ++mb)
#pragma unroll
    for (int rr = 0; rr < 16; ++rr) tmax = fmaxf(tmax, s[mb][rr]);
  return swap_halves_max(tmax) * scale_log2;
}

// ... the lazy move of the reference max (with the rescale of numerator and sum) ...
__device__ __forceinline__ void softmax_rescale(f32x16 (&o)[4], float& m_i, float& l_i, float tm) {
  if (__builtin_amdgcn_ballot_w64(tm > m_i + kLazyLog2) != 0) {
    const float m_new = fmaxf(m_i, tm);
    const float alpha = m_new == -INFINITY ? 1.f : exp2_fast(m_i - m_new);  // 0 when m_i = -inf
    m_i = m_new;
    l_i *= alpha;
#pragma unroll
    for (int md = 0; md < 4; ++md)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) o[md][rr] *= alpha;
  }
}

// The row sum l from the bf16 p that the P.V product uses (16 v_dot2 per row block and tile
// instead of 32 fp32 adds): numerator and denominator then weigh every key alike. Measured
// interleaved: steady batch 693.6 -> 680.2 us, cfg3 prefill 95.9 -> 95.4 us.
#ifndef PK_PREFILL_DOT_SUM
#define PK_PREFILL_DOT_SUM 1
#endif
// ... and the exponentials against the reference max, packed to bf16 as the P.V B operand.
template <int NB>
__device__ __forceinline__ void softmax_exp(f32x16 (&s)[NB], bf16x8 (&pb)[2 * NB], float m_i, float& l_i,
                                            float scale_log2) {
  const float m_use = (m_i == -INFINITY) ? 0.f : m_i;  // row saw no key yet: every p is 0
  float psum = 0.f;
#pragma unroll
  for (int mb = 0; mb < NB; ++mb)
#pragma unroll
    for (int rr = 0; rr < 16; ++rr) {
      const float p = exp2_fast(__builtin_fmaf(s[mb][rr], scale_log2, -m_use));
      s[mb][rr] = p;
      if (!PK_PREFILL_DOT_SUM) psum += p;
    }
  // B operand of k-block kb2: element e of lane half `half` stands for key
  // 16 kb2 + 8 (e >> 2) + 4 half + (e & 3) = accumulator element 8 (kb2 & 1) + e of
  // half-tile kb2 >> 1.
#pragma unroll
  for (int kb2 = 0; kb2 < 2 * NB; ++kb2)
#pragma unroll
    for (int e = 0; e < 8; ++e) pb[kb2][e] = static_cast<__bf16>(s[kb2 >> 1][8 * (kb2 & 1) + e]);
  if (PK_PREFILL_DOT_SUM) {
    // the row sum from the bf16 p the P.V product uses: one v_dot2 per pair of keys
    const bf16x2 one = {static_cast<__bf16>(1.f), static_cast<__bf16>(1.f)};
#pragma unroll
    for (int kb2 = 0; kb2 < 2 * NB; ++kb2)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const bf16x2 pr = {pb[kb2][e], pb[kb2][e + 1]};
        psum = __builtin_amdgcn_fdot2_f32_bf16(pr, one, psum, false);
      }
  }
  l_i += psum;
}

__device__ __forceinline__ void softmax_block(f32x16 (&s)[2], f32x16 (&o)[4], bf16x8 (&pb)[4], float& m_i, float& l_i,
                                              int t0, int lim, bool full, float scale_log2, int half) {
  const float tm = full ? softmax_max<2, false>(s, t0, lim, scale_log2, half)
                        : softmax_max<2, true>(s, t0, lim, scale_log2, half);
  softmax_rescale(o, m_i, l_i, tm);
  softmax_exp<2>(s, pb, m_i, l_i, scale_log2);
}

// Per-lane LDS byte offsets of the MFMA operand reads inside a stage.
//   K, k-block kb: row col (+ 32 for the second half-tile: + 8 KiB), chunk 2 kb + half,
//     swizzled with col & 15 (32 mb + col has the same low bits);
//   V, d-block md: row 4 half + (src >> 2) (+ 16 kb2 rows: + 4 KiB, + 8 rows: + 2 KiB), the
//     swizzle (2 r) & 15 does not see those row steps.
struct TileLanes {
  int k0, v0;
  // Offsets of k-block kb and d-block md: the k-block moves the chunk by 2 kb and the d-block
  // by 4 md, bits the swizzles only XOR with lane bits, so the offsets are k0 ^ 32 kb and
  // v0 ^ 64 md (one VALU op per read instead of twelve live registers).
  __device__ __forceinline__ int k(int kb) const { return k0 ^ (32 * kb); }
  __device__ __forceinline__ int v(int md) const { return v0 ^ (64 * md); }
};

__device__ __forceinline__ TileLanes tile_lanes(int lane) {
  TileLanes t;
  const int col = lane & 31;
  const int half = lane >> 5;
  const int grp = lane >> 4;
  const int src = lane & 15;
  t.k0 = col * kRowBytes + k_slot(col, half) * 16;
  const int d = 16 * (grp & 1) + 4 * (src & 3);
  const int r = 4 * half + (src >> 2);
  t.v0 = r * kRowBytes + v_slot(r, d >> 3) * 16 + (d & 7) * 2;
  return t;
}

// One 64-key tile for the wavefront's kRowBlocks blocks of 32 query rows.
__device__ __forceinline__ void compute_tile(const lds_char* sK, const lds_char* sV, const TileLanes& tl,
                                             const bf16x8 (&qb)[kRowBlocks][kHeadDim / 16],
                                             f32x16 (&o)[kRowBlocks][4], float (&m_i)[kRowBlocks],
                                             float (&l_i)[kRowBlocks], int t0, const int (&lim)[kRowBlocks],
                                             const bool (&full)[kRowBlocks], float scale_log2, int lane) {
  const int half = lane >> 5;
  f32x16 s[kRowBlocks][2];
#pragma unroll
  for (int rb = 0; rb < kRowBlocks; ++rb)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) s[rb][mb][rr] = 0.f;
  // K A operand of half-tile mb, k-block kb: read kKDepth k-blocks ahead of the MFMAs that
  // use it, the order pinned by scheduling groups (the compiler's own schedule read each
  // k-block right before its two MFMAs and waited for it: no read was in flight while an
  // MFMA ran).
#ifndef PK_PREFILL_KDEPTH
#define PK_PREFILL_KDEPTH 2
#endif
  constexpr int kKDepth = PK_PREFILL_KDEPTH;
  constexpr int kKBlocks = kHeadDim / 16;
  bf16x8 ka[kKBlocks][2];
  const auto read_k = [&](int kb) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
      ka[kb][mb] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>(sK + tl.k(kb) +
                                                                                   mb * 32 * kRowBytes);
  };
#pragma unroll
  for (int kb = 0; kb < kKDepth; ++kb) read_k(kb);
#pragma unroll
  for (int kb = 0; kb < kKBlocks; ++kb) {
    if (kb + kKDepth < kKBlocks) read_k(kb + kKDepth);
#pragma unroll
    for (int rb = 0; rb < kRowBlocks; ++rb)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
        s[rb][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[kb][mb], qb[rb][kb], s[rb][mb], 0, 0, 0);
  }
#pragma unroll
  for (int kb = 0; kb < kKDepth; ++kb) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // DS reads
#pragma unroll
  for (int kb = 0; kb < kKBlocks; ++kb) {
    if (kb + kKDepth < kKBlocks) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 2 * kRowBlocks, 0);  // MFMAs
  }

  bf16x8 pb[kRowBlocks][4];
#pragma unroll
  for (int rb = 0; rb < kRowBlocks; ++rb)
    softmax_block(s[rb], o[rb], pb[rb], m_i[rb], l_i[rb], t0, lim[rb], full[rb], scale_log2, half);

  // O^T += V^T . P^T over 16-key k-blocks. The A operand (4 consecutive keys of one
  // head_dim element, twice) comes from the row-major V tile through the LDS transpose
  // read: in each 16-lane group, source lane s addresses 4 elements of key row
  // key0 + (s >> 2) at head_dim d0 + 4 (s & 3), and lane i receives element d0 + i of keys
  // key0 .. key0 + 3. Each A operand serves every row block.
#pragma unroll
  for (int kb2 = 0; kb2 < 4; ++kb2) {
#pragma unroll
    for (int md = 0; md < 4; ++md) {
      const lds_char* p_lo = sV + tl.v(md) + kb2 * 16 * kRowBytes;
      const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          const_cast<lds_v4i16*>(reinterpret_cast<const lds_v4i16*>(p_lo)));
      const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          const_cast<lds_v4i16*>(reinterpret_cast<const lds_v4i16*>(p_lo + 8 * kRowBytes)));
      const bf16x8 av = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
      for (int rb = 0; rb < kRowBlocks; ++rb)
        o[rb][md] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, pb[rb][kb2], o[rb][md], 0, 0, 0);
    }
  }
}

// Sequence geometry shared by the plan, prefill and merge kernels.
struct SeqDims {
  int q0, Lq, k0, Lk, P, nq;  // nq: query tiles of the sequence (0: not a prefill sequence)
};

template <int TM>
__device__ __forceinline__ SeqDims seq_dims(const AttnArgs& a, int b) {
  SeqDims d;
  d.q0 = a.cu_q[b];
  d.Lq = a.cu_q[b + 1] - d.q0;
  d.k0 = a.cu_k[b];
  d.Lk = min(a.cu_k[b + 1] - d.k0, a.max_seqlen_k);
  d.P = d.Lk - d.Lq;
  // Lq == 1 rows belong to the decode kernel; Lq <= 0 or Lk <= 0 is graph padding
  d.nq = (d.Lq <= 1 || d.Lk <= 0) ? 0 : min((d.Lq + TM - 1) / TM, a.prefill_qtiles);
  return d;
}

// Key tiles query tile qt needs: keys below its last row's causal limit.
template <int TM, bool CAUSAL>
__device__ __forceinline__ int unit_tiles(const SeqDims& d, int qt) {
  const int kv_end = CAUSAL ? min(d.Lk, (qt + 1) * TM + d.P) : d.Lk;
  return kv_end > 0 ? (kv_end + kTileKeys - 1) / kTileKeys : 0;
}

// Splits of a unit of t tiles for split size T, and the start tile of split s.
__device__ __forceinline__ int unit_splits(int t, int T) { return t > T ? (t + T - 1) / T : 1; }
__device__ __forceinline__ int split_begin(int t, int n, int s) { return (int)((unsigned)(t * s) / (unsigned)n); }

// Length bucket of a group of t tiles (0 = longest) of N buckets for split size T.
template <int N>
__device__ __forceinline__ int length_bucket(int t, int T) {
  int j = 0;  // the largest j < N with t N > j T (compares, no division)
#pragma unroll
  for (int i = 1; i < N; ++i) j = t * N > i * T ? i : j;
  return N - 1 - j;
}

// Work list. Waves take sequences in turn and lanes take a sequence's query tiles, so a
// long prompt's tiles are planned in parallel. Groups land in their length bucket through
// LDS cursors: the order inside a bucket depends on timing, but a group's work and the
// merge order of its splits do not, so results are bit-identical from run to run.
template <int G, bool CAUSAL, bool SMALL>
__global__ __launch_bounds__(kPlanThreads) void prefill_plan_kernel(const AttnArgs a) {
  constexpr int TM = kPrefillRows / G;
  constexpr int W = kPlanThreads / kWave;
  constexpr int kBuckets = SMALL ? kSmallBuckets : kLargeBuckets;
  __shared__ long long red[W];
  __shared__ int cur[kBuckets + 2];  // bucket cursors, partial-group cursor, merge cursor
  // (sequence, Lq, Lk) of the prefill sequences among the first kPlanCache, in any order: the
  // passes read them from LDS and do not walk the decode rows of a mixed batch (128 of them beside
  // 8 chunks: nine rounds of the wavefronts per pass instead of one, 9.5 us for the plan). SMALL:
  // all of them, in their own places (the list's barrier and atomics cost a small call 1 us)
  __shared__ int4 dims[kPlanCache];
  __shared__ int listed;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int S = a.num_seqs;
  const int hkv = a.num_kv_heads;

  if constexpr (!SMALL) {
    if (tid == 0) listed = 0;
    __syncthreads();
  }
  for (int b = tid; b < min(S, kPlanCache); b += kPlanThreads) {
    const SeqDims d = seq_dims<TM>(a, b);
    if constexpr (SMALL)
      dims[b] = make_int4(b, d.Lq, d.Lk, 0);
    else if (d.nq > 0)
      dims[atomicAdd(&listed, 1)] = make_int4(b, d.Lq, d.Lk, 0);
  }
  __syncthreads();
  const int nlist = SMALL ? min(S, kPlanCache) : listed;
  const int nseq = nlist + max(0, S - kPlanCache);  // entries of the passes: the list, then the rest
  auto dims_of = [&](int i, int& b) {
    if (i >= nlist) {
      b = kPlanCache + i - nlist;
      return seq_dims<TM>(a, b);
    }
    SeqDims d;
    d.q0 = d.k0 = 0;  // not used by the plan
    const int4 e = dims[i];
    b = e.x;
    d.Lq = e.y;
    d.Lk = e.z;
    d.P = d.Lk - d.Lq;
    d.nq = (d.Lq <= 1 || d.Lk <= 0) ? 0 : min((d.Lq + TM - 1) / TM, a.prefill_qtiles);
    return d;
  };

  // pass 1: total key tiles over all units
  long long tiles = 0;
  for (int i = wave; i < nseq; i += W) {
    int b;
    const SeqDims d = dims_of(i, b);
    for (int qt = lane; qt < d.nq; qt += kWave) tiles += unit_tiles<TM, CAUSAL>(d, qt);
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) tiles += __shfl_xor(tiles, o, kWave);
  if (lane == 0) red[wave] = tiles;
  if (tid < kBuckets + 2) cur[tid] = 0;
  __syncthreads();
  long long work = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) work += red[w];
  work *= hkv;
  // split size: kSplitNum / kSplitDen of the work per slot, at least kMinSplitTiles (no unit
  // has 2^20 tiles)
  const int T = (int)min((long long)(1 << 20),
                         max((long long)kMinSplitTiles,
                             (kSplitNum * (work / kSplitDen) + a.pf_slots - 1) / a.pf_slots + 1));

  // pass 2: groups per length bucket
  for (int i = wave; i < nseq; i += W) {
    int b;
    const SeqDims d = dims_of(i, b);
    for (int qt = lane; qt < d.nq; qt += kWave) {
      const int t = unit_tiles<TM, CAUSAL>(d, qt);
      const int n = unit_splits(t, T);
      for (int sp = 0; sp < n; ++sp)
        atomicAdd(&cur[length_bucket<kBuckets>(split_begin(t, n, sp + 1) - split_begin(t, n, sp), T)], 1);
    }
  }
  __syncthreads();
  int tot = 0, start[kBuckets];
#pragma unroll
  for (int k = 0; k < kBuckets; ++k) {
    start[k] = tot;
    tot += cur[k];
  }
  __syncthreads();
  if (tid < kBuckets) cur[tid] = 0;
  __syncthreads();

  // pass 3: emit one entry per group; kv heads are expanded by index (item i = head i % hkv
  // of group i / hkv)
  for (int i = wave; i < nseq; i += W) {
    int b;
    const SeqDims d = dims_of(i, b);
    for (int qt = lane; qt < d.nq; qt += kWave) {
      const int t = unit_tiles<TM, CAUSAL>(d, qt);
      const int n = unit_splits(t, T);
      // partial groups stay below 3 x slots / hkv (each split unit has more than T tiles)
      const int pg = n > 1 ? atomicAdd(&cur[kBuckets], n) : -1;
      for (int sp = 0; sp < n; ++sp) {
        const int tb = split_begin(t, n, sp);
        const int te = split_begin(t, n, sp + 1);
        const int k = length_bucket<kBuckets>(te - tb, T);
        const int grp = start[k] + atomicAdd(&cur[k], 1);
        if (grp < a.pf_item_cap) a.pf_items[grp] = make_int4(b, qt, tb | (te << 16), n > 1 ? pg + sp : -1);
      }
      if (n > 1) {
        const int m = atomicAdd(&cur[kBuckets + 1], 1);
        if (m < a.pf_merge_cap) a.pf_merges[m] = make_int4(b, qt, pg, n);
      }
    }
  }
  // LDS-only: the counts in cur are final; the work-list stores need not complete before the
  // queue header's (the prefill kernel, a later launch, reads both)
  lds_barrier();
  // sub-queue x starts behind the items that its work-groups take without a claim
  if (tid < 8) a.pf_queue[tid * kPrefillQueueStride] = (a.pf_slots - tid + 7) / 8;
  if (tid == 0) {
    a.pf_queue[kPrefillQueueMeta] = (int)(min((int64_t)tot, (int64_t)a.pf_item_cap) * hkv);
    a.pf_queue[kPrefillQueueMeta + 1] = (int)(min((int64_t)cur[kBuckets + 1], (int64_t)a.pf_merge_cap) * hkv);
    a.pf_queue[kPrefillQueueMeta + 2] = T;
  }
}

// ---- Claims and item inputs, of both prefill kernels -----------------------------------------
// Wavefront 0: the claimed index, or -1 once every sub-queue is exhausted (own: the work-group's own
// sub-queue xcd may have items left; pend: what lane 0's claim on it returned). Stealing reads the
// other seven counters at once (lanes 0..6) and takes from the first sub-queue after this one
// that has items left; a claim that lost the race reads again. Counters only grow, so a stale
// read never shows a sub-queue exhausted too early.
__device__ __forceinline__ int claim_finish(const AttnArgs& a, int xcd, int num_items, int lane, bool& own, int pend) {
  if (own) {
    const int64_t cand = (int64_t)__builtin_amdgcn_readfirstlane(pend) * 8 + xcd;
    if (cand < num_items) return (int)cand;
    own = false;
  }
  for (;;) {
    const int q = (xcd + 1 + lane) & 7;
    const int c = lane < 7 ? __hip_atomic_load(&a.pf_queue[q * kPrefillQueueStride], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT)
                           : 0;
    const uint64_t left = __builtin_amdgcn_ballot_w64(lane < 7 && (int64_t)c * 8 + q < num_items);
    if (left == 0) return -1;
    const int qs = (xcd + 1 + __builtin_ctzll(left)) & 7;
    int r = 0;
    if (lane == 0) r = atomicAdd(&a.pf_queue[qs * kPrefillQueueStride], 1);
    const int64_t cand = (int64_t)__builtin_amdgcn_readfirstlane(r) * 8 + qs;
    if (cand < num_items) return (int)cand;
  }
}
// Item i's work-list group (lanes 0..3), sequence b's bounds (lanes 0..3: cu_q[b], cu_q[b + 1], cu_k[b],
// cu_k[b + 1]) and its first 64 block-table entries (one per lane: a tile's block id is a readlane).
__device__ __forceinline__ int load_group(const AttnArgs& a, int i, int lane) {
  return lane < 4 ? reinterpret_cast<const int*>(a.pf_items)[(int64_t)(i / a.num_kv_heads) * 4 + lane] : 0;
}
__device__ __forceinline__ int load_bounds(const AttnArgs& a, int b, int lane) {
  const int32_t* p = lane < 2 ? a.cu_q + b + lane : a.cu_k + b + (lane - 2);
  return lane < 4 ? *p : 0;
}
template <bool PAGED>
__device__ __forceinline__ int load_bt(const AttnArgs& a, int b, int lane) {
  if constexpr (!PAGED) return 0;
  return lane < min(a.bt_stride, kWave) ? a.block_table[(int64_t)b * a.bt_stride + lane] : 0;
}

// ---- Small calls ---------------------------------------------------------------------------
// Eight wavefronts of one row block each (two per SIMD) in phases QK - softmax - PV per 64-key
// tile, K and V through registers into two LDS stages. Its tile takes half as long again as
// prefill_kernel's, but an item starts sooner (no pipeline to fill, a third of the code to fetch
// into a cold instruction cache), which decides where a work-group has one or two short items:
// one item of 7 tiles per work-group 36.7 against 40.9 us a call, 15 chunks of 100 over 2048
// keys 74.5 against 81.0. prefill_kernel is ahead from about 34 tiles per work-group (see
// small_prefill).
constexpr int kW8Stages = 2;             // K and V LDS stages

// One work item: kv head g of group `it` = (sequence b, query tile qt, key tiles [tb, te),
// partial group or -1). The caller's hooks run at three points, which the kernel uses to
// claim and prefetch the next item: last_step when the last key tile starts, after_tiles
// after the last tile's barrier (before the epilogue), after_epilogue after its stores.
template <int G, bool PAGED, bool CAUSAL, class LastStep, class AfterTiles, class AfterEpilogue>
__device__ __forceinline__ void prefill_item_w8(const AttnArgs& a, const int4 it, const int g, const int cuv,
                                             const int bt_lane, lds_char* const (&KS)[kW8Stages],
                                             lds_char* const (&VS)[kW8Stages],
                                             int wave, int lane,
                                             LastStep&& last_step, AfterTiles&& after_tiles,
                                             AfterEpilogue&& after_epilogue) {
  constexpr int D = kHeadDim;
  constexpr int TN = kTileKeys;
  constexpr int TM = kPrefillRows / G;
  static_assert(TM >= 32, "a 32-row block is one head");
  const int b = it.x;
  const int qt = it.y;
  const int tb = it.z & 0xffff;
  const int te = it.z >> 16;
  const int part = it.w < 0 ? -1 : it.w * a.num_kv_heads + g;
  // The work list is trusted only as far as the buffers reach: an entry naming a sequence or
  // key tiles outside this call (a workspace overwritten by an overlapping call) is skipped.
  // The hooks run in every case, so the work-group's barriers and claims stay in step.
  // cuv (lanes 0..3) holds the sequence's bounds, loaded by the caller.
  const int q0 = __builtin_amdgcn_readlane(cuv, 0);
  const int Lq = __builtin_amdgcn_readlane(cuv, 1) - q0;
  const int k0 = __builtin_amdgcn_readlane(cuv, 2);
  const int Lk = min(__builtin_amdgcn_readlane(cuv, 3) - k0, a.max_seqlen_k);
  const int P = Lk - Lq;
  if (b < 0 || b >= a.num_seqs || Lq <= 0 || tb > te || te > (Lk + TN - 1) / TN) {
    lds_barrier();
    after_tiles();
    after_epilogue();
    return;
  }
  const int tok_begin = qt * TM;

  const int col = lane & 31;   // MFMA column = this lane's query row inside a block
  const int half = lane >> 5;
  int row[kRowBlocks], h[kRowBlocks], tok[kRowBlocks], lim[kRowBlocks], lim_lo[kRowBlocks], lim_hi[kRowBlocks];
#pragma unroll
  for (int rb = 0; rb < kRowBlocks; ++rb) {
    const int r0 = (wave * kRowBlocks + rb) * 32;  // first row of the block: 32 tokens of one head
    row[rb] = r0 + col;
    h[rb] = g * G + row[rb] / TM;
    tok[rb] = tok_begin + row[rb] % TM;
    lim[rb] = CAUSAL ? min(Lk - 1, tok[rb] + P) : Lk - 1;  // last key this row sees
    const int blo = tok_begin + r0 % TM;
    lim_lo[rb] = CAUSAL ? min(Lk - 1, blo + P) : Lk - 1;       // keys <= lim_lo: seen by all rows
    lim_hi[rb] = CAUSAL ? min(Lk - 1, blo + 31 + P) : Lk - 1;  // keys >  lim_hi: seen by none
  }

  // Q^T B operands: k-block kb covers d in [16 kb, 16 kb + 16); lane holds 8 of them.
  // Rows past Lq read the last row (finite) and are never stored.
  bf16x8 qb[kRowBlocks][D / 16];
#pragma unroll
  for (int rb = 0; rb < kRowBlocks; ++rb) {
    const uint16_t* qp = a.q + (int64_t)(q0 + min(tok[rb], Lq - 1)) * a.q_row_stride + h[rb] * D + 8 * half;
#pragma unroll
    for (int kb = 0; kb < D / 16; ++kb)
      qb[rb][kb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp + kb * 16));
  }
  f32x16 o[kRowBlocks][4];
  float m_i[kRowBlocks], l_i[kRowBlocks];
#pragma unroll
  for (int rb = 0; rb < kRowBlocks; ++rb) {
#pragma unroll
    for (int md = 0; md < 4; ++md)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) o[rb][md][rr] = 0.f;
    m_i[rb] = -INFINITY;
    l_i[rb] = 0.f;
  }

  // Pipeline, one barrier per tile: at step n, tile n + 1 (registers) is written to stage
  // (n + 1) & 1 and the loads of tile n + 2 go out into the same registers, tile n is computed
  // from stage n & 1, and the barrier publishes tile n + 1.
  const int ntiles = te - tb;
  const int tbase = tb * TN;
  const LoadLanes ll = load_lanes(a, wave, lane, kTileKeys);
  const TileLanes tl = tile_lanes(lane);
  KvRegs R;
  // The tile loop is entered only from the path that stored tile 0, whose register wait also
  // covers the Q loads issued before it. (With a path around that store into the loop, the
  // compiler's wait counting assumed the Q loads could still be in flight in every iteration
  // and made each k-block's QK MFMA wait for the global loads issued before it -- tile n + 2's
  // staging loads -- exposing their latency in every tile.)
  if (ntiles <= 0) {
    lds_barrier();
  } else {
    load_tile_regs<PAGED>(a, b, k0, Lk, g, bt_lane, wave, lane, tbase, ll, R);
    store_tile_lds(R, KS[0], VS[0], wave, lane);
    if (ntiles > 1) load_tile_regs<PAGED>(a, b, k0, Lk, g, bt_lane, wave, lane, tbase + TN, ll, R);
    lds_barrier();
    for (int n0 = 0; n0 < ntiles; n0 += 2) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int n = n0 + s;
        if (n >= ntiles) break;
        if (n == ntiles - 1) last_step();
        const int t0 = tbase + n * TN;
        // tile n + 1 (loaded during tile n - 1) goes to the other stage -- last read at step
        // n - 1, before the previous barrier -- and its registers take tile n + 2's loads: one
        // set of staging registers (a second set, holding tile n + 2 while tile n + 1 waited to
        // be stored after tile n, took the kernel to 256 VGPRs with spills; 2.4% slower)
        if (n + 1 < ntiles) {
          store_tile_lds(R, KS[s ^ 1], VS[s ^ 1], wave, lane);
          if (n + 2 < ntiles) load_tile_regs<PAGED>(a, b, k0, Lk, g, bt_lane, wave, lane, t0 + 2 * TN, ll, R);
        }
        bool any = false, full[kRowBlocks];
#pragma unroll
        for (int rb = 0; rb < kRowBlocks; ++rb) {
          any |= t0 <= lim_hi[rb];
          full[rb] = t0 + TN - 1 <= lim_lo[rb];
        }
        if (any) compute_tile(KS[s], VS[s], tl, qb, o, m_i, l_i, t0, lim, full, a.scale_log2, lane);
        lds_barrier();
      }
    }
  }

  after_tiles();
  // Epilogue: O^T element rr of d-block md is d = 32 md + 8 (rr >> 2) + 4 half + (rr & 3).
#pragma unroll
  for (int rb = 0; rb < kRowBlocks; ++rb) {
    const float l_tot = swap_halves_sum(l_i[rb]);
    if (tok[rb] >= Lq) continue;
    if (part < 0) {
      const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;  // a row that saw no key is written as 0
      uint16_t* op = a.out + (int64_t)(q0 + tok[rb]) * a.out_row_stride + h[rb] * D + 4 * half;
#pragma unroll
      for (int md = 0; md < 4; ++md)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
          uint2 w;
          w.x = pack_bf16x2(o[rb][md][4 * gq] * inv, o[rb][md][4 * gq + 1] * inv);
          w.y = pack_bf16x2(o[rb][md][4 * gq + 2] * inv, o[rb][md][4 * gq + 3] * inv);
          *reinterpret_cast<uint2*>(op + md * 32 + 8 * gq) = w;
        }
    } else if (part < a.pf_part_cap) {
      // The split's own output o / l in bf16 -- as precise as an unsplit row's output -- with
      // (max, sum) in fp32 for the merge. Chunk-major (chunk = 4 dims = d / 4): one store
      // instruction writes two contiguous 256-byte runs (32 rows x 8 bytes per lane half).
      const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
      uint16_t* po = a.pf_part_o + (int64_t)part * (32 * kPrefillRows * 4);
#pragma unroll
      for (int md = 0; md < 4; ++md)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
          const int chunk = 8 * md + 2 * gq + half;
          uint2 w;
          w.x = pack_bf16x2(o[rb][md][4 * gq] * inv, o[rb][md][4 * gq + 1] * inv);
          w.y = pack_bf16x2(o[rb][md][4 * gq + 2] * inv, o[rb][md][4 * gq + 3] * inv);
          *reinterpret_cast<uint2*>(po + ((int64_t)chunk * kPrefillRows + row[rb]) * 4) = w;
        }
      if (half == 0)
        *reinterpret_cast<float2*>(a.pf_part_ml + ((int64_t)part * kPrefillRows + row[rb]) * 2) =
            make_float2(m_i[rb], l_tot);
    }
  }
  after_epilogue();
}

template <int G, bool PAGED, bool CAUSAL>
__global__ __launch_bounds__(kPrefillThreads, kWavesPerSimd) void prefill_w8_kernel(const AttnArgs a) {
  // two stages per operand (constant stage indices put the stage offset in immediates)
  __shared__ __attribute__((aligned(1024))) char sK[kW8Stages][kTileBytes];
  __shared__ __attribute__((aligned(1024))) char sV[kW8Stages][kTileBytes];
  __shared__ int s_item;  // the claimed item index
  lds_char* KS[kW8Stages];
  lds_char* VS[kW8Stages];
#pragma unroll
  for (int st = 0; st < kW8Stages; ++st) {
    KS[st] = (lds_char*)sK[st];
    VS[st] = (lds_char*)sV[st];
  }

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // Work-groups are dealt to the 8 XCDs round-robin by linear id: this one claims items of
  // sub-queue x = blockIdx mod 8 (items i = 8 j + x, counter x) while it has any, then steals
  // from the others. Wavefront 0 claims; lane 0 owns the atomics.
  const int xcd = blockIdx.x & 7;
  const int num_items = (int)min((int64_t)a.pf_queue[kPrefillQueueMeta], (int64_t)a.pf_item_cap * a.num_kv_heads);
  // The claim on the own sub-queue goes out when the current item starts its last key tile,
  // so the atomic overlaps that tile and the work-group holds no item it cannot start yet
  // (items are long: a claim made earlier would hold one back from idle work-groups at the
  // end). `pend` is that atomic's result (lane 0).
  bool own = true;
  int pend = 0;
  const auto claim_issue = [&]() {
    if (wave == 0 && own && lane == 0) pend = atomicAdd(&a.pf_queue[xcd * kPrefillQueueStride], 1);
  };
  // The next item's inputs load in two dependent steps around the current item's epilogue:
  // its work-list group (lanes 0..3) before the epilogue's stores, then the sequence's
  // bounds (lanes 0..3: cu_q[b], cu_q[b + 1], cu_k[b], cu_k[b + 1]) and first 64
  // block-table entries (one per lane: a tile's block id is a readlane, not a dependent
  // global load) after them.
  // The work list is trusted only as far as the buffers reach: a group naming a sequence
  // outside this call (a workspace overwritten by an overlapping call) reads sequence 0's
  // bounds and is skipped by prefill_item_w8.
  const auto seq_of = [&](int grpv) {
    const int b = __builtin_amdgcn_readlane(grpv, 0);
    return b >= 0 && b < a.num_seqs ? b : 0;
  };
  // the first item is the work-group's own (item blockIdx), as in prefill_kernel
  int idx = (int)blockIdx.x < num_items ? (int)blockIdx.x : -1;
  int grpv = 0, cuv = 0, btv = 0;
  if (idx >= 0) {
    grpv = load_group(a, idx, lane);
    cuv = load_bounds(a, seq_of(grpv), lane);
    btv = load_bt<PAGED>(a, seq_of(grpv), lane);
  }
  while (idx >= 0) {
    int next = -1, next_grpv = 0, next_cuv = 0, next_btv = 0;
    bool claimed = false;
    const int grp = idx / a.num_kv_heads;
    const int4 it = make_int4(__builtin_amdgcn_readlane(grpv, 0), __builtin_amdgcn_readlane(grpv, 1),
                              __builtin_amdgcn_readlane(grpv, 2), __builtin_amdgcn_readlane(grpv, 3));
    prefill_item_w8<G, PAGED, CAUSAL>(
        a, it, idx - grp * a.num_kv_heads, cuv, btv, KS, VS, wave, lane,
        [&]() {
          claim_issue();
          claimed = true;
        },
        [&]() {
          // s_item was last read before this item's first barrier
          if (wave == 0) {
            if (!claimed) claim_issue();
            const int c = claim_finish(a, xcd, num_items, lane, own, pend);
            if (lane == 0) s_item = c;
          }
          lds_barrier();
          next = __builtin_amdgcn_readfirstlane(s_item);
          if (next >= 0) next_grpv = load_group(a, next, lane);
        },
        [&]() {
          if (next >= 0) {
            next_cuv = load_bounds(a, seq_of(next_grpv), lane);
            next_btv = load_bt<PAGED>(a, seq_of(next_grpv), lane);
          }
        });
    idx = next;
    grpv = next_grpv;
    cuv = next_cuv;
    btv = next_btv;
  }
}

// ---- The prefill kernel's tile loop --------------------------------------------------------
// What bounds the other kernel's loop (eight wavefronts of one row block, phases QK - softmax - PV
// with a barrier per tile, for 2048 cycles of MFMA per 64-key tile): the two wavefronts of
// a SIMD pass the phases together, so the MFMA, vector and LDS work add up, and every
// wavefront reads the whole tile from LDS (256 KiB per tile and CU at 128 B per cycle: as long as
// the MFMAs). Two row blocks per wavefront halve the LDS reads, and one wavefront per SIMD has
// the registers (O 128, Q 64, two steps' scores 64 and P 32) to run three steps' parts beside
// each other. What the loop then needs, measured per instruction (cycles, one wavefront): an MFMA
// takes 32, up to five independent vector instructions beside it are free, a sixth and further
// ones cost 4-5, a vector instruction that uses the previous one's result 8, an exponential 8,
// v_dot2 (which the MFMA pipe executes too) 17, an LDS read beside a full slot 4. Hence: no
// instruction uses a result of its own slot; sums by a small MFMA, not v_dot2; no running max (one
// reference per row and item with 2^120 of room, checked by the sum at the end); K and V bypass
// the registers. 16 chunks of 1024 over 4096-token prefixes (618 GFLOP), item starts and ends
// included: 4982 -> 4160 cycles per tile, MFMA pipes busy 43.6 -> 55.8% (counters), 650-671 -> 587-625 us
// per call with the 24 us store, at a clock that falls with the load (1.93 GHz, less after several
// such calls): an 8192^3 matrix product of the vendor's library reaches 1.21 PFLOP/s here. Short items
// are bound by their start and end, so calls of few tiles keep the other kernel (small_prefill).
constexpr int kPfWaves = 4;                      // one wavefront per SIMD, 64 query rows each
constexpr int kPfThreads = kPfWaves * kWave;
constexpr int kPfRB = kPrefillRows / (32 * kPfWaves);  // 32-row blocks per wavefront
// LDS: four K and three V stages; the stages that an item's first loads do not use (K 3, V 1, V 2)
// and one tile more hold its Q rows on their way to registers, and a last tile the output rows on
// their way out.
constexpr int kLdsK0 = 0, kLdsK1 = kTileBytes, kLdsK2 = 2 * kTileBytes, kLdsK3 = 4 * kTileBytes;
constexpr int kLdsV0 = 3 * kTileBytes, kLdsV1 = 5 * kTileBytes, kLdsV2 = 6 * kTileBytes;
constexpr int kLdsQ = 4 * kTileBytes, kLdsO = 8 * kTileBytes;
constexpr int kPfLdsBytes = 9 * kTileBytes;
constexpr int kPfAhead = 3;                      // operands read this many ahead of their MFMAs
constexpr int kStepKeys = 32;                    // keys per pipeline step (half a tile)
constexpr int kPfLoads = kTileKeys / kPfWaves / 4;     // 16-byte loads per lane, operand and tile
constexpr float kSumLimit = 1.329227995784916e36f;  // 2^120: the largest row sum of one reference

static_assert(kPfLoads == 4, "stage_tile issues four loads per operand");

// Byte offsets of the tile rows this lane moves (row r clamped to `last`), for stage_tile.
template <bool V>
__device__ __forceinline__ void stage_offsets(int row_stride, int wave, int lane, int last, int (&off)[kPfLoads]) {
  const int slot = lane & 15;
#pragma unroll
  for (int i = 0; i < kPfLoads; ++i) {
    const int r = 4 * kPfLoads * wave + 4 * i + (lane >> 4);
    const int c = V ? v_chunk(r, slot) : slot ^ (r & 15);
    off[i] = (min(r, last) * row_stride + c * 8) * 2 + 1024 * (kPfLoads - 1 - i);
  }
}

// The wavefront's rows of a tile, memory to LDS without registers: lane l of load i moves 16
// bytes from base + off[i] - 1024 (3 - i) to lds + 1024 i + 16 l. (The instruction's offset
// moves both addresses; off carries the correction.)
__device__ __forceinline__ void stage_tile(const char* base, const int (&off)[kPfLoads], int lds) {
  const uint64_t u = (uint64_t)(base - 1024 * (kPfLoads - 1));
  const uint64_t b = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32;
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %5\n\t"
      "global_load_lds_dwordx4 %2, %5 offset:1024\n\t"
      "global_load_lds_dwordx4 %3, %5 offset:2048\n\t"
      "global_load_lds_dwordx4 %4, %5 offset:3072"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(b)
      : "m0", "memory");
}

// One of stage_tile's loads.
template <int I>
__device__ __forceinline__ void stage_load(const char* base, int off, int lds) {
  const uint64_t u = (uint64_t)(base - 1024 * (kPfLoads - 1));
  const uint64_t b = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32;
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2 offset:%c3"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(off), "s"(b), "i"(1024 * I)
      : "m0", "memory");
}

// 16 bytes per lane from per-lane addresses to lds + 16 l.
__device__ __forceinline__ void load_lds16(const uint16_t* src, int lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(src)
      : "m0", "memory");
}

// Waits until at most N of this wavefront's vector memory operations are in flight.
template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// The wavefront's state over an item. O and the second row block's Q live in accumulation
// registers, everything else in architectural ones.
struct PfState {
  bf16x8 q[kPfRB][kHeadDim / 16];
  f32x16 o[kPfRB][4];
  f32x16 s[2][kPfRB];          // scores of steps of either parity
  u32x4 p[2][kPfRB][2];        // P (bf16 pairs) of steps of either parity
  bf16x8 kf[kPfAhead];         // K operands read ahead
  float nm[kPfRB];             // minus the reference max of the exponentials
  u32x2 ones;                  // four 1.0 in bf16
  f32x4 ls[kPfRB];             // the tile loops' row sums over this lane's keys (four equal values)
  float l[kPfRB];              // the item's
};

__device__ __forceinline__ bf16x8 read_k(const lds_char* sK, const TileLanes& tl, int kb) {
  return *reinterpret_cast<const __attribute__((address_space(3))) bf16x8*>(sK + tl.k(kb));
}
__device__ __forceinline__ bf16x8 read_v(const lds_char* sV, const TileLanes& tl, int f) {
  const lds_char* p = sV + tl.v(f & 3) + (f >> 2) * 16 * kRowBytes;
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      const_cast<lds_v4i16*>(reinterpret_cast<const lds_v4i16*>(p)));
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      const_cast<lds_v4i16*>(reinterpret_cast<const lds_v4i16*>(p + 8 * kRowBytes)));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}
// The MFMAs are written out because the compiler keeps one register kind per kernel for their
// results: S, which the vector instructions read, belongs in architectural registers and O, which
// nothing reads before the item's end, in accumulation registers. The compiler does not add the
// wait states of an MFMA that it does not know, so the order of the stream provides them: a score
// is read 16 MFMAs after the last that wrote it, P is used 16 MFMAs after its conversion, K, Q
// and V operands come from LDS reads (which are waited for); pf_iteration's scheduling barriers
// keep that order, and tests/test_prefill_stream.py checks it in the built code.
// S += K Q^T with S in architectural registers, Q in architectural (row block 0) or accumulation
// registers (row block 1).
__device__ __forceinline__ void mfma_s(f32x16& s, const bf16x8& k, const bf16x8& q, bool first, int rb) {
  if (first && rb == 0)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "v"(q));
  else if (first)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "a"(q));
  else if (rb == 0)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "v"(q));
  else
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "a"(q));
}

// O += V^T P^T with O in accumulation registers.
__device__ __forceinline__ void mfma_o(f32x16& o, const bf16x8& v, const u32x4& p) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(o) : "v"(v), "v"(p));
}

// Row sums += the four keys of p (ones times P^T, 4 x 4 x 4 in 16 blocks: a lane's result is the sum of
// its own four). The sums take the rounded P of the P.V product, so that numerator and denominator
// weigh every key alike: a key far above the others gives its V row exactly, where a sum of the
// unrounded p is off by up to 2^-9. Issued right before a slot's large MFMA it costs the 8 cycles that it
// runs and saves the additions: 16 chunks of 1024 over 4096-token prefixes 584 (unrounded sums) -> 591
// us; after the large MFMA, where it holds up the vector instructions, 600; unpacking the rounded
// pairs for vector additions 609.
__device__ __forceinline__ void mfma_sum(f32x4& l, const u32x2& ones, const u32x2& p) {
  asm volatile("v_mfma_f32_4x4x4_16b_bf16 %0, %1, %2, %0" : "+a"(l) : "a"(ones), "v"(p));
}

// The first softmax of an item (step 0): the reference is the row's max over the first tile's keys, whose
// scores are both here; P = 2^(s - reference) in bf16. Later steps keep the reference: the row's largest
// p is 1 or more, so products with small V rows stay as far from fp32's smallest numbers as with a
// running max. (The max's own p is exactly 1. With the first step's max alone the largest p of short
// rows was rounded more often: error against 64 bits of fresh prompts 2.008e-3, with the tile's 1.991e-3.)
__device__ __forceinline__ void softmax_first(PfState& st, int t0, const int (&lim)[kPfRB], float scale_log2,
                                              int half) {
#pragma unroll
  for (int rb = 0; rb < kPfRB; ++rb) {
    float s[16];
    float t = -INFINITY;
#pragma unroll
    for (int rr = 0; rr < 16; ++rr) {
      const int key = t0 + 8 * (rr >> 2) + 4 * half + (rr & 3);
      s[rr] = key > lim[rb] ? -INFINITY : st.s[0][rb][rr];
      t = fmaxf(t, fmaxf(s[rr], key + kStepKeys > lim[rb] ? -INFINITY : st.s[1][rb][rr]));
    }
    t = swap_halves_max(t) * scale_log2;
    const float nm = t == -INFINITY ? 0.f : -t;
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const float p0 = exp2_fast(__builtin_fmaf(s[i], scale_log2, nm));
      const float p1 = exp2_fast(__builtin_fmaf(s[i + 1], scale_log2, nm));
      const bf16x2 pr = {static_cast<__bf16>(p0), static_cast<__bf16>(p1)};
      st.p[0][rb][i >> 3][(i & 7) >> 1] = __builtin_bit_cast(uint32_t, pr);
    }
    st.nm[rb] = nm;
  }
}

// Pipeline iteration i of a wavefront: S(i + 1) = K Q^T of step i + 1, the softmax of step i and
// O += V^T P^T of step i - 1, three independent streams; CUR = i & 1. 32 slots of one MFMA each
// (16 QK, then 16 PV), and beside it the slot's share of the LDS reads (kPfAhead operands ahead;
// the next iteration's first K operands at the end), of the softmax and, with STAGE, of the loads
// of a tile (from `src`, offsets `soff`, to LDS `lds`). MASK: keys past a row's limit count 0.
template <int CUR, bool MASK, bool STAGE>
__device__ __forceinline__ void pf_iteration(PfState& st, const lds_char* sK, const lds_char* sKn, const lds_char* sV,
                                             const TileLanes& tl, int t0, const int (&lim)[kPfRB],
                                             float scale_log2, int half, const char* src,
                                             const int (&soff)[kPfLoads], int lds) {
  constexpr int NXT = CUR ^ 1;
  constexpr int KB = kHeadDim / 16;
  constexpr int NE = 16 * kPfRB;  // scores per lane
  bf16x8 kf[KB], vf[8];
  float x[NE];  // a score on its way to p
#pragma unroll
  for (int j = 0; j < kPfAhead; ++j) kf[j] = st.kf[j];
  // elements started by the end of slot s: 32 of them in 29 slots, so the last is packed in slot 31
  const auto nf = [](int s) { return s < 0 ? 0 : (s + 1) * NE >= 29 * NE ? NE : ((s + 1) * NE + 28) / 29; };
#pragma unroll
  for (int sl = 0; sl < 32; ++sl) {
    // LDS reads
    if (sl < 16 && (sl & 1) == 0 && sl / 2 + kPfAhead < KB)
      kf[sl / 2 + kPfAhead] = read_k(sK, tl, sl / 2 + kPfAhead);
    const int f = sl - (16 - 2 * kPfAhead);
    if (f >= 0 && (f & 1) == 0 && f / 2 < 8) vf[f / 2] = read_v(sV, tl, f / 2);
    const int j = sl - (29 - kPfAhead);
    if (j >= 0 && j < kPfAhead) st.kf[j] = read_k(sKn, tl, j);
    // the tile's loads, between the others
    if constexpr (STAGE) {
      if (sl == 3) stage_load<0>(src, soff[0], lds);
      if (sl == 7) stage_load<1>(src, soff[1], lds);
      if (sl == 11) stage_load<2>(src, soff[2], lds);
      if (sl == 15) stage_load<3>(src, soff[3], lds);
    }
    // MFMAs
    if (sl < 16) {
      if (sl & 1) {  // the sum of step i - 1, row block 1's last keys (packed in slot 31) at the end
        const u32x4 p = st.p[NXT][sl >> 3][(sl >> 2) & 1];
        mfma_sum(st.ls[sl >> 3], st.ones, (sl & 2) ? u32x2{p[2], p[3]} : u32x2{p[0], p[1]});
      }
      mfma_s(st.s[NXT][sl & 1], kf[sl / 2], st.q[sl & 1][sl / 2], sl < 2, sl & 1);
    } else {
      const int fv = (sl - 16) / 2, rb = sl & 1;
      mfma_o(st.o[rb][fv & 3], vf[fv], st.p[NXT][rb][fv >> 2]);
    }
    // softmax: the scale and reference of some elements, the exponentials of those of the slot
    // before, packing of those of the slot before that
#pragma unroll
    for (int e = nf(sl - 4); e < nf(sl - 3); ++e) {
      if (e & 1) {
        const bf16x2 pr = {static_cast<__bf16>(x[e - 1]), static_cast<__bf16>(x[e])};
        st.p[CUR][e >> 4][(e & 15) >> 3][(e & 7) >> 1] = __builtin_bit_cast(uint32_t, pr);
      }
    }
#pragma unroll
    for (int e = nf(sl - 1); e < nf(sl); ++e) {
      const int rr = e & 15, rb = e >> 4;
      float v = st.s[CUR][rb][rr];
      if constexpr (MASK) v = t0 + 8 * (rr >> 2) + 4 * half + (rr & 3) > lim[rb] ? -INFINITY : v;
      x[e] = __builtin_fmaf(v, scale_log2, st.nm[rb]);
    }
#pragma unroll
    for (int e = nf(sl - 2); e < nf(sl - 1); ++e) {
      x[e] = exp2_fast(x[e]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int rb = 0; rb < kPfRB; ++rb) {
    // S is final here (the MFMAs that wrote it are 16 MFMAs back), and P is computed before here
    asm volatile("" : "+v"(st.s[NXT][rb]), "+v"(st.p[CUR][rb][0]), "+v"(st.p[CUR][rb][1]));
  }
}

// Cursor over an item's key tiles: the tile's first K and V row of kv head g and its first key.
template <bool PAGED>
struct TileCursor {
  const char *k, *v;
  int t0, last, j, off;
  int64_t kstep, vstep;
  __device__ __forceinline__ void to_block(const AttnArgs& a, int b, int g, int bt_lane) {
    const int blk = j < kWave ? __builtin_amdgcn_readlane(bt_lane, j)
                              : __builtin_amdgcn_readfirstlane(a.block_table[(int64_t)b * a.bt_stride + j]);
    k = reinterpret_cast<const char*>(a.k + (int64_t)blk * a.k_block_stride + (int64_t)off * a.k_row_stride +
                                      g * kHeadDim);
    v = reinterpret_cast<const char*>(a.v + (int64_t)blk * a.v_block_stride + (int64_t)off * a.v_row_stride +
                                      g * kHeadDim);
  }
  __device__ __forceinline__ void init(const AttnArgs& a, int b, int g, int k0, int tbase, int ntiles, int bt_lane) {
    t0 = tbase;
    last = tbase + (ntiles - 1) * kTileKeys;
    kstep = a.k_row_stride * (2 * kTileKeys);
    vstep = a.v_row_stride * (2 * kTileKeys);
    j = off = 0;
    k = reinterpret_cast<const char*>(a.k + g * kHeadDim);
    v = reinterpret_cast<const char*>(a.v + g * kHeadDim);
    if constexpr (PAGED) {
      j = tbase / a.block_size;  // block_size % 64 == 0: a tile sits inside one block
      off = tbase - j * a.block_size;
      if (ntiles > 0) to_block(a, b, g, bt_lane);
    } else {
      k += (int64_t)(k0 + tbase) * a.k_row_stride * 2;
      v += (int64_t)(k0 + tbase) * a.v_row_stride * 2;
    }
  }
  // To the next tile; the last one stays.
  __device__ __forceinline__ void advance(const AttnArgs& a, int b, int g, int bt_lane) {
    if (t0 < last) step(a, b, g, bt_lane);
  }
  __device__ __forceinline__ void step(const AttnArgs& a, int b, int g, int bt_lane) {
    t0 += kTileKeys;
    k += kstep;
    v += vstep;
    if constexpr (PAGED) {
      off += kTileKeys;
      if (off == a.block_size) {
        off = 0;
        ++j;
        to_block(a, b, g, bt_lane);
      }
    }
  }
};

// The first row of row block rb of wavefront `wave`. A wavefront's two blocks hold the same tokens
// of two heads where the unit has two heads (G > 1), so that the causal limit crosses few of its
// steps; G = 1: neighbouring tokens.
template <int G>
__device__ __forceinline__ int block_row(int wave, int rb) {
  constexpr int NB = kPrefillRows / G / 32;  // blocks of a head
  return 32 * (NB == 8 ? 2 * wave + rb : wave % NB + NB * rb + 2 * NB * (wave / NB));
}


// A work item: kv head g of group (sequence b, query tile qt, key tiles [tb, te), partial group),
// with the sequence's bounds.
struct PfItem {
  int b, qt, tb, te, part, g, q0, Lq, k0, Lk;
};

// From the work-list entry and the sequence's bounds (cu_q[b], cu_q[b + 1], cu_k[b], cu_k[b + 1]).
// The work list is trusted only as far as the buffers reach: an entry naming a sequence or key
// tiles outside this call (a workspace overwritten by an overlapping call) becomes an item
// without rows or tiles.
__device__ __forceinline__ PfItem make_item(const AttnArgs& a, int idx, const int4& grp, const int4& cu) {
  PfItem it;
  it.g = __builtin_amdgcn_readfirstlane(idx % a.num_kv_heads);
  it.b = grp.x;
  it.qt = grp.y;
  it.tb = grp.z & 0xffff;
  it.te = grp.z >> 16;
  it.part = grp.w < 0 ? -1 : grp.w * a.num_kv_heads + it.g;
  it.q0 = cu.x;
  it.Lq = cu.y - cu.x;
  it.k0 = cu.z;
  it.Lk = min(cu.w - cu.z, a.max_seqlen_k);
  if (it.b < 0 || it.b >= a.num_seqs || it.Lq <= 0 || it.tb > it.te ||
      it.te > (it.Lk + kTileKeys - 1) / kTileKeys) {
    it.b = it.qt = it.tb = it.te = it.q0 = it.Lq = it.k0 = it.Lk = 0;
    it.part = -1;
  }
  return it;
}

// v, as a value of its own at every use: what is computed from it is computed again for every item
// instead of being kept in registers through the tile loops.
__device__ __forceinline__ int per_item(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// An item's tiles one after the other with a running row max (numerator and sum rescaled when it
// moves by more than 2^kLazyLog2): what an item takes whose scores leave the range that one
// reference covers. A row block leaves out the steps that none of its rows sees (their p is 0, but a V
// row of infinities or NaN would reach O as 0 * infinity). Ends with a barrier.
template <int G, bool PAGED, bool CAUSAL>
__device__ __forceinline__ void prefill_item_safe(const AttnArgs& a, PfState& st, const PfItem& it, int bt_lane,
                                                  const int (&lim)[kPfRB], lds_char* const smem, int wave, int lane) {
  constexpr int TM = kPrefillRows / G;
  const int b = it.b, g = it.g, k0 = it.k0, Lk = it.Lk, tbase = it.tb * kTileKeys, ntiles = it.te - it.tb;
  const int half = lane >> 5;
  int lim_hi[kPfRB];  // the last key that a row of the block sees
  // Q again (the tile loops' operands need not outlive them)
#pragma unroll
  for (int rb = 0; rb < kPfRB; ++rb) {
    const int row = block_row<G>(wave, rb) + (lane & 31);
    const int blo = it.qt * TM + block_row<G>(wave, rb) % TM;
    lim_hi[rb] = CAUSAL ? min(Lk - 1, blo + 31 + Lk - it.Lq) : Lk - 1;
    const int tok = min(it.qt * TM + row % TM, it.Lq - 1);
    const uint16_t* qp = a.q + (int64_t)(it.q0 + tok) * a.q_row_stride + (g * G + row / TM) * kHeadDim + 8 * half;
#pragma unroll
    for (int kb = 0; kb < kHeadDim / 16; ++kb)
      st.q[rb][kb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp + kb * 16));
  }
  const TileLanes tl = tile_lanes(lane);
  const int lds0 = (int)(uintptr_t)smem + 4 * kPfLoads * wave * kRowBytes;
  TileCursor<PAGED> cur;
  cur.init(a, b, g, k0, tbase, ntiles, bt_lane);
  float m[kPfRB];
  const float zero = __int_as_float(per_item(0));
#pragma unroll
  for (int rb = 0; rb < kPfRB; ++rb) {
    m[rb] = -INFINITY;
    st.l[rb] = 0.f;
#pragma unroll
    for (int md = 0; md < 4; ++md)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) st.o[rb][md][rr] = zero;
  }
#pragma unroll 1
  for (int n = 0; n < ntiles; ++n) {
    const int t0 = cur.t0;
    int off[kPfLoads];
    stage_offsets<false>((int)a.k_row_stride, wave, lane, min(kTileKeys, Lk - 1 - t0), off);
    stage_tile(cur.k, off, lds0);
    stage_offsets<true>((int)a.v_row_stride, wave, lane, min(kTileKeys, Lk - 1 - t0), off);
    stage_tile(cur.v, off, lds0 + kTileBytes);
    cur.advance(a, b, g, bt_lane);
    wait_vm<0>();
    lds_barrier();
#pragma unroll 1
    for (int hs = 0; hs < 2; ++hs) {
      const lds_char* const sK = smem + hs * 32 * kRowBytes;
      const lds_char* const sV = smem + kTileBytes + hs * 32 * kRowBytes;
#pragma unroll
      for (int rb = 0; rb < kPfRB; ++rb) {
        if (t0 + hs * kStepKeys > lim_hi[rb]) continue;
        f32x16 s[1];
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) s[0][rr] = 0.f;
#pragma unroll
        for (int kb = 0; kb < kHeadDim / 16; ++kb)
          s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_k(sK, tl, kb), st.q[rb][kb], s[0], 0, 0, 0);
        bf16x8 pb[2];
        const float tm = softmax_max<1, true>(s, t0 + hs * kStepKeys, lim[rb], a.scale_log2, half);
        softmax_rescale(st.o[rb], m[rb], st.l[rb], tm);
        softmax_exp<1>(s, pb, m[rb], st.l[rb], a.scale_log2);
#pragma unroll
        for (int f = 0; f < 8; ++f)
          st.o[rb][f & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_v(sV, tl, f), pb[f >> 2], st.o[rb][f & 3],
                                                                     0, 0, 0);
      }
    }
    lds_barrier();
  }
#pragma unroll
  for (int rb = 0; rb < kPfRB; ++rb) st.nm[rb] = -m[rb];
}

template <int G, bool PAGED, bool CAUSAL>
__global__ __launch_bounds__(kPfThreads, 1) void prefill_kernel(const AttnArgs a) {
  constexpr int D = kHeadDim;
  constexpr int TN = kTileKeys;
  constexpr int TM = kPrefillRows / G;
  static_assert(TM >= 32, "a 32-row block is one head");
  __shared__ __attribute__((aligned(1024))) char smem_[kPfLdsBytes];
  __shared__ int s_item;  // the claimed item index
  __shared__ int s_redo;  // the current item needs a running max
  lds_char* const smem = (lds_char*)smem_;
  __attribute__((address_space(3))) int* const redo = (__attribute__((address_space(3))) int*)&s_redo;

  const int tid = threadIdx.x;
  const int lane_ = tid & (kWave - 1), lane = lane_;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // Work-groups are dealt to the 8 XCDs round-robin by linear id: this one claims items of
  // sub-queue x = blockIdx mod 8 (items i = 8 j + x, counter x) while it has any, then steals
  // from the others. Wavefront 0 claims; lane 0 owns the atomics.
  const int xcd = blockIdx.x & 7;
  const int num_items = (int)min((int64_t)a.pf_queue[kPrefillQueueMeta], (int64_t)a.pf_item_cap * a.num_kv_heads);
  bool own = true;
  int pend = 0;  // lane 0 of wavefront 0: the claim's result
  const auto claim_issue = [&]() {
    if (wave == 0 && own && lane == 0) {
      // the address as a per-lane value keeps the compiler from combining the wavefront's lanes
      // and waiting for the result here
      int z = 0;
      asm volatile("" : "+v"(z));
      pend = atomicAdd(&a.pf_queue[xcd * kPrefillQueueStride + z], 1);
    }
  };
  // The next item's inputs, in three steps over the current item's last tiles, each begun at the
  // top of a tile and ended at its bottom, so that none of the dependent round trips is waited
  // out: 0 the claim, published by wavefront 0; 1 the work-list entry; 2 the sequence's bounds
  // and block-table entries. What is kept between tiles is uniform or has arrived.
  int next = -1, gv = 0, cv = 0, btn = 0;
  int4 ng = make_int4(0, 0, 0, 0), nc = make_int4(0, 0, 0, 0);
  const auto next_begin = [&](int s) {
    if (s == 0) {
      claim_issue();
    } else if (s == 1) {
      next = __builtin_amdgcn_readfirstlane(s_item);
      if (next >= 0) gv = load_group(a, next, lane);
    } else if (s == 2 && next >= 0) {
      const int b = ng.x >= 0 && ng.x < a.num_seqs ? ng.x : 0;  // see make_item
      cv = load_bounds(a, b, lane);
      btn = load_bt<PAGED>(a, b, lane);
    }
  };
  const auto lanes4 = [&](int v) {
    return make_int4(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 1), __builtin_amdgcn_readlane(v, 2),
                     __builtin_amdgcn_readlane(v, 3));
  };
  const auto next_end = [&](int s) {
    if (s == 0) {
      if (wave == 0) {
        const int c = claim_finish(a, xcd, num_items, lane, own, pend);
        if (lane == 0) s_item = c;
      }
    } else if (s == 1) {
      if (next >= 0) ng = lanes4(gv);
    } else if (s == 2 && next >= 0) {
      nc = lanes4(cv);
      asm volatile("" : "+v"(btn));
    }
  };

  const int col = lane & 31;   // MFMA column = this lane's query row inside a block
  const int half = lane >> 5;
  const TileLanes tl = tile_lanes(lane);
  const int wrow = 4 * kPfLoads * wave * kRowBytes;  // this wavefront's rows of a stage
  const int lds0 = (int)(uintptr_t)smem;

  // The first item is the work-group's own (item blockIdx): no claim, and its work-list entry
  // loads with the item count (the list has room for more groups than there are work-groups).
  next = (int)blockIdx.x;
  ng = lanes4(load_group(a, next, lane));
  if (next >= num_items) return;
  next_begin(2);
  next_end(2);
  PfItem it = make_item(a, next, ng, nc);
  int btv = btn;

  // The start of an item: its Q operands and its first tiles (K 0, K 1, V 0, K 2) are requested.
  // V lags K by two tiles: v1 and v2 are the K cursor's last two positions.
  TileCursor<PAGED> cur;
  int koff[kPfLoads], voff[kPfLoads];
  const char *v1, *v2;
  const auto clamp_k = [&]() {
    if (cur.t0 + TN > it.Lk)
      stage_offsets<false>((int)a.k_row_stride, wave, per_item(lane_), it.Lk - 1 - cur.t0, koff);
  };
  const auto stage_v = [&](const char* src, int t, int lds) {
    if (t + TN > it.Lk) stage_offsets<true>((int)a.v_row_stride, wave, per_item(lane_), it.Lk - 1 - t, voff);
    stage_tile(src, voff, lds);
  };
  const auto start_item = [&]() {
    const int lane = per_item(lane_);
    // Q rows (row r of the wavefront's 64, 16-byte chunk c in slot c ^ (r & 15), as K tiles are
    // stored); rows past Lq take the last row (finite) and are never stored.
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 4 * i + (lane >> 4);
      const int row0 = block_row<G>(wave, i >> 3);
      const int tok = max(0, min(it.qt * TM + row0 % TM + (r & 31), it.Lq - 1));
      load_lds16(a.q + (int64_t)(it.q0 + tok) * a.q_row_stride + (it.g * G + row0 / TM) * D + ((lane & 15) ^ (r & 15)) * 8,
                 lds0 + kLdsQ + wave * 64 * kRowBytes + i * 1024);
    }
    const int ntiles = it.te - it.tb, tbase = it.tb * TN;
    cur.init(a, it.b, it.g, it.k0, tbase, ntiles, btv);
    if (ntiles <= 0) return;
    stage_offsets<false>((int)a.k_row_stride, wave, lane, kTileKeys, koff);
    stage_offsets<true>((int)a.v_row_stride, wave, lane, kTileKeys, voff);
    clamp_k();
    stage_tile(cur.k, koff, lds0 + kLdsK0 + wrow);
  };
  const auto start_rest = [&]() {
    const int ntiles = it.te - it.tb, tbase = it.tb * TN;
    if (ntiles <= 0) return;
    const char* const vfirst = cur.v;
    cur.advance(a, it.b, it.g, btv);
    clamp_k();
    v1 = cur.v;
    stage_tile(cur.k, koff, lds0 + kLdsK1 + wrow);
    stage_v(vfirst, tbase, lds0 + kLdsV0 + wrow);
    cur.advance(a, it.b, it.g, btv);
    clamp_k();
    v2 = cur.v;
    stage_tile(cur.k, koff, lds0 + kLdsK2 + wrow);
    cur.advance(a, it.b, it.g, btv);
    clamp_k();
  };
  start_item();
  start_rest();

  for (;;) {
    PfState st;
    const int ntiles = it.te - it.tb, tbase = it.tb * TN;
    const int P = it.Lk - it.Lq;
    int lim[kPfRB];
    int lim_lo = 0x7fffffff, lim_hi = -1;  // keys <= lim_lo: seen by all the wavefront's rows, > lim_hi: by none
    int lim_hi0 = -1;                      // > lim_hi0: by none of the first block's
#pragma unroll
    for (int rb = 0; rb < kPfRB; ++rb) {
      const int r0 = block_row<G>(wave, rb);  // 32 tokens of one head
      const int blo = it.qt * TM + r0 % TM;
      // last key of the item this row sees
      lim[rb] = min(it.te * TN, CAUSAL ? min(it.Lk, blo + col + P + 1) : it.Lk) - 1;
      lim_lo = min(lim_lo, CAUSAL ? min(it.Lk - 1, blo + P) : it.Lk - 1);
      lim_hi = max(lim_hi, CAUSAL ? min(it.Lk - 1, blo + 31 + P) : it.Lk - 1);
      if (rb == 0) lim_hi0 = lim_hi;
      st.nm[rb] = 0.f;
    }
    const auto clear_o = [&]() {
      st.ones = u32x2{0x3f803f80u, 0x3f803f80u};
      asm volatile("" : "+a"(st.ones));
#pragma unroll
      for (int rb = 0; rb < kPfRB; ++rb) {
        st.ls[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(st.ls[rb]));
#pragma unroll
        for (int md = 0; md < 4; ++md) {
          const float zero = __int_as_float(per_item(0));
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) st.o[rb][md][rr] = zero;
          asm volatile("" : "+a"(st.o[rb][md]));
        }
      }
    };
    // steps (32 keys) this wavefront's rows see
    const int nw = min(2 * ntiles, (lim_hi - tbase + kStepKeys) >> 5);

    // everything start_item requested is here; Q^T B operands: k-block kb covers d in
    // [16 kb, 16 kb + 16), a lane holds 8 of them
    wait_vm<0>();
    const int qrow = per_item(kLdsQ + wave * 64 * kRowBytes);
#pragma unroll
    for (int rb = 0; rb < kPfRB; ++rb)
#pragma unroll
      for (int kb = 0; kb < D / 16; ++kb)
        st.q[rb][kb] = read_k(smem + qrow + rb * 32 * kRowBytes, tl, kb);
#pragma unroll
    for (int kb = 0; kb < D / 16; ++kb) {
      asm volatile("" : "+v"(st.q[0][kb]));
      asm volatile("" : "+a"(st.q[1][kb]));
    }
    next = -1;
    if (ntiles < 2) {  // no tile to put the claim in
      next_begin(0);
      next_end(0);
    }
    lds_barrier();
    if (threadIdx.x == 0) *redo = 0;  // last read before this barrier, next written after a later one
    if (ntiles <= 0) {
      next_begin(1);
      next_end(1);
      next_begin(2);
      next_end(2);
      clear_o();
    } else {
      clear_o();
      int k0s = kLdsK0, k1s = kLdsK1, k2s = kLdsK2, k3s = kLdsK3;  // K tiles n .. n + 3
      int v1s = kLdsV2, v0s = kLdsV0, vns = kLdsV1;                // V tiles n - 1 .. n + 1
      // Body n: loads of K tile n + 3 and V tile n + 1; K tile n + 2 and V tile n land by its end.
      const auto stage = [&](int n) {
        if (n + 1 < ntiles) stage_v(v1, tbase + (n + 1) * TN, lds0 + vns + wrow);
        v1 = v2;
        v2 = cur.v;
        if (n + 3 < ntiles) stage_tile(cur.k, koff, lds0 + k3s + wrow);
        cur.advance(a, it.b, it.g, btv);
        clamp_k();
        next_begin(n + 2 - ntiles);
      };
      const auto rotate = [&]() {
        const int k = k0s;
        k0s = k1s;
        k1s = k2s;
        k2s = k3s;
        k3s = k;
        const int v = v1s;
        v1s = v0s;
        v0s = vns;
        vns = v;
      };
      const auto finish = [&](int n) {
        next_end(n + 2 - ntiles);
        if (n == ntiles) return;
        if (n + 3 < ntiles)
          wait_vm<8>();
        else if (n + 1 < ntiles)
          wait_vm<4>();
        else
          wait_vm<0>();
        lds_barrier();
        rotate();
      };
      // body 0: the scores of steps 0 and 1, the first softmax
      stage(0);
      if (nw > 0) {
        bf16x8 k[16];
#pragma unroll
        for (int j = 0; j < kPfAhead; ++j) k[j] = read_k(smem + k0s, tl, j);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int f = j + kPfAhead;
          if (f < 16)
            k[f] = read_k(smem + k0s + (f >> 3) * 32 * kRowBytes, tl, f & 7);
          else
            st.kf[f - 16] = read_k(smem + k1s, tl, f - 16);
#pragma unroll
          for (int rb = 0; rb < kPfRB; ++rb) mfma_s(st.s[j >> 3][rb], k[j], st.q[rb][j & 7], (j & 7) == 0, rb);
          __builtin_amdgcn_sched_barrier(0);
        }
        // the wait states between an MFMA and a VALU read of its result
        asm volatile("s_nop 15\n\ts_nop 7"
                     : "+v"(st.s[0][0]), "+v"(st.s[0][1]), "+v"(st.s[1][0]), "+v"(st.s[1][1]));
        softmax_first(st, tbase, lim, a.scale_log2, half);
      } else {  // not used; defined, so that no register carries the last item's through this one
#pragma unroll
        for (int rb = 0; rb < kPfRB; ++rb) {
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) st.s[0][rb][rr] = st.s[1][rb][rr] = 0.f;
          st.p[0][rb][0] = st.p[0][rb][1] = u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int j = 0; j < kPfAhead; ++j) st.kf[j] = st.q[0][0];
      }
      finish(0);
      int t0 = tbase + kStepKeys;  // first key of step 2n - 1
      int n = 1;
      // what the allocator put aside over body 0 comes back before the loop, not in it (its waits
      // would count the loop's own loads)
#pragma unroll
      for (int rb = 0; rb < kPfRB; ++rb)
        asm volatile("" : "+v"(st.s[1][rb]), "+v"(st.p[0][rb][0]), "+v"(st.p[0][rb][1]), "+v"(st.nm[rb]));
#pragma unroll 1
      for (; t0 + TN - 1 <= lim_lo && n + 4 < ntiles; ++n, t0 += TN) {
        const lds_char* const ks = smem + k0s;
        const lds_char* const vs = smem + v1s;
        pf_iteration<1, false, true>(st, ks, ks + 32 * kRowBytes, vs, tl, t0, lim, a.scale_log2, half, v1, voff,
                                     lds0 + vns + wrow);
        pf_iteration<0, false, true>(st, ks + 32 * kRowBytes, smem + k1s, vs + 32 * kRowBytes, tl, t0 + kStepKeys, lim,
                                     a.scale_log2, half, cur.k, koff, lds0 + k3s + wrow);
        v1 = v2;
        v2 = cur.v;
        cur.step(a, it.b, it.g, btv);
        wait_vm<8>();
        lds_barrier();
        rotate();
      }
      clamp_k();
#pragma unroll 1
      for (; t0 + TN - 1 <= lim_lo && n < ntiles; ++n, t0 += TN) {
        stage(n);
        const lds_char* const ks = smem + k0s;
        const lds_char* const vs = smem + v1s;
        pf_iteration<1, false, false>(st, ks, ks + 32 * kRowBytes, vs, tl, t0, lim, a.scale_log2, half, nullptr, koff, 0);
        pf_iteration<0, false, false>(st, ks + 32 * kRowBytes, smem + k1s, vs + 32 * kRowBytes, tl, t0 + kStepKeys,
                                      lim, a.scale_log2, half, nullptr, koff, 0);
        finish(n);
      }
#pragma unroll 1
      for (; n <= ntiles; ++n, t0 += TN) {
        stage(n);
        if (2 * n - 2 < nw) {
          const lds_char* const ks = smem + k0s;
          const lds_char* const vs = smem + v1s;
          pf_iteration<1, true, false>(st, ks, ks + 32 * kRowBytes, vs, tl, t0, lim, a.scale_log2, half, nullptr, koff,
                                       0);
          pf_iteration<0, true, false>(st, ks + 32 * kRowBytes, smem + k1s, vs + 32 * kRowBytes, tl, t0 + kStepKeys,
                                       lim, a.scale_log2, half, nullptr, koff, 0);
        }
        finish(n);
      }
    }
    // The sum shows whether the item's reference held: a row whose scores rose beyond the limit (or
    // that overflowed on the way), or that never reached its reference (first keys of -infinity leave
    // it at 0, wherever the others lie), has the whole item done again with a running max. So has one
    // whose O is not finite where the sum is above what a running max could have left (p up to
    // 2^kLazyLog2 for every key): large V rows overflow there beside sums within the limit.
    float l_tot[kPfRB];
    bool bad = false, large = false;
#pragma unroll
    for (int rb = 0; rb < kPfRB; ++rb) {
      asm volatile("" : "+a"(st.ls[rb]));
      st.l[rb] = st.ls[rb][0];
      l_tot[rb] = swap_halves_sum(st.l[rb]);
      bad |= !(l_tot[rb] <= kSumLimit) || (l_tot[rb] < 0.5f && lim[rb] >= tbase);
      large |= l_tot[rb] > (float)(TN << (int)kLazyLog2) * (float)ntiles;
    }
    // With one head per unit a wavefront's second block may see a tile that its first does not, whose V
    // rows reach the first's O as 0 * V: the same look for what is not finite.
    if constexpr (G == 1) large |= ntiles > 0 && tbase + (nw - 1) / 2 * TN > lim_hi0;
    if (__builtin_amdgcn_ballot_w64(large) != 0) {
      float z = 0.f;  // NaN if any is not finite
#pragma unroll
      for (int rb = 0; rb < kPfRB; ++rb)
#pragma unroll
        for (int md = 0; md < 4; ++md) {
          asm volatile("" : "+a"(st.o[rb][md]));
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) z = __builtin_fmaf(st.o[rb][md][rr], 0.f, z);
        }
      bad |= z != 0.f;
    }
    if (ntiles > 0 && __builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) *redo = 1;
    lds_barrier();  // every wavefront is done with the item's tiles
    if (__builtin_expect(ntiles > 0 && __builtin_amdgcn_readfirstlane(*redo) != 0, 0)) {
      prefill_item_safe<G, PAGED, CAUSAL>(a, st, it, btv, lim, smem, wave, per_item(lane_));
#pragma unroll
      for (int rb = 0; rb < kPfRB; ++rb) l_tot[rb] = swap_halves_sum(st.l[rb]);
    }
    // the next item's first loads go out before this one's results are written
    const PfItem done = it;
    if (next >= 0) {
      it = make_item(a, next, ng, nc);
      btv = btn;
      start_item();
    }
    // O^T element rr of d-block md is d = 32 md + 8 (rr >> 2) + 4 half + (rr & 3).
    const int lane = per_item(lane_), col = lane & 31, half = lane >> 5;
    float inv[kPfRB];
#pragma unroll
    for (int rb = 0; rb < kPfRB; ++rb) {
      inv[rb] = l_tot[rb] > 0.f ? 1.f / l_tot[rb] : 0.f;  // a row that saw no key is written as 0
#pragma unroll
      for (int md = 0; md < 4; ++md) asm volatile("" : "+a"(st.o[rb][md]));
    }
    if (done.part < 0) {
      // Through LDS, so that a store covers 128 consecutive bytes of a row (straight from the
      // accumulators it would cover 16): 64 dims of a row block in 4 KiB, 16-byte chunk c of row r
      // in slot c ^ (r & 7). The four pieces take this wavefront's rows of the stages that its
      // second batch of loads fills, which goes out after they are read.
      const auto piece = [&](int p) { return smem + (p == 0 ? kLdsO : p == 1 ? kLdsK1 : p == 2 ? kLdsK2 : kLdsV0) + wrow; };
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const f32x16& o = st.o[p >> 1][2 * (p & 1) + (c >> 2)];
          const float iv = inv[p >> 1];
          u32x2 w;
          w[0] = pack_bf16x2(o[4 * (c & 3)] * iv, o[4 * (c & 3) + 1] * iv);
          w[1] = pack_bf16x2(o[4 * (c & 3) + 2] * iv, o[4 * (c & 3) + 3] * iv);
          *reinterpret_cast<__attribute__((address_space(3))) u32x2*>(piece(p) + col * 128 + ((c ^ (col & 7)) << 4) +
                                                                      half * 8) = w;
        }
      u32x4 w[4][4];
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 8 * i + (lane >> 3);
          w[p][i] = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(
              piece(p) + r * 128 + (((lane & 7) ^ (r & 7)) << 4));
        }
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(w[p][i]));
      if (next >= 0) start_rest();
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int row0 = block_row<G>(wave, p >> 1);
        const int tok0 = done.qt * TM + row0 % TM + (lane >> 3);
        uint16_t* op = a.out + (int64_t)(done.q0 + tok0) * a.out_row_stride + (done.g * G + row0 / TM) * D +
                       64 * (p & 1) + 8 * (lane & 7);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (tok0 + 8 * i < done.Lq) *reinterpret_cast<u32x4*>(op + 8 * i * a.out_row_stride) = w[p][i];
      }
    } else {
      if (next >= 0) start_rest();
#pragma unroll
      for (int rb = 0; rb < kPfRB; ++rb) {
        const int row = block_row<G>(wave, rb) + col;
        const int tok = done.qt * TM + row % TM;
        if (done.part >= a.pf_part_cap || tok >= done.Lq) continue;
        // The split's own output o / l in bf16 -- as precise as an unsplit row's output -- with
        // (reference, sum) in fp32 for the merge. Chunk-major (chunk = 4 dims = d / 4): one store
        // instruction writes two contiguous 256-byte runs (32 rows x 8 bytes per lane half).
        uint16_t* po = a.pf_part_o + (int64_t)done.part * (32 * kPrefillRows * 4);
#pragma unroll
        for (int md = 0; md < 4; ++md)
#pragma unroll
          for (int gq = 0; gq < 4; ++gq) {
            const int chunk = 8 * md + 2 * gq + half;
            uint2 w;
            w.x = pack_bf16x2(st.o[rb][md][4 * gq] * inv[rb], st.o[rb][md][4 * gq + 1] * inv[rb]);
            w.y = pack_bf16x2(st.o[rb][md][4 * gq + 2] * inv[rb], st.o[rb][md][4 * gq + 3] * inv[rb]);
            *reinterpret_cast<uint2*>(po + ((int64_t)chunk * kPrefillRows + row) * 4) = w;
          }
        // The merge takes 2^(reference - largest reference) as a split's scale, so the reference has
        // to be near the row's max: the sum's exponent, far from 0 here, moves into it.
        if (half == 0) {
          const float e = (float)__builtin_amdgcn_frexp_expf(l_tot[rb]);
          *reinterpret_cast<float2*>(a.pf_part_ml + ((int64_t)done.part * kPrefillRows + row) * 2) =
              make_float2(l_tot[rb] > 0.f ? e - st.nm[rb] : -INFINITY, __builtin_amdgcn_frexp_mantf(l_tot[rb]));
        }
      }
    }
    if (next < 0) return;
  }
}

// Merge the partials of every split unit: out = sum_s w_s o_s / sum_s w_s with
// w_s = exp2(m_s - max_s m_s) l_s, o_s the split's normalised output (bf16), m_s a reference that
// is near the split's largest score, so that a weight that flushes to 0 is negligible. Work item =
// (split unit, quarter of head_dim, kv head); thread t owns row t of the unit and 8 chunks
// of 4 dims. At most 4 wavefronts per SIMD: the register budget lets the loads of
// kMergeLoads splits be in flight at once. Two rounds of loads reach the first store: the
// work-list entry (the first one read together with the work count, from a list slot that
// always exists), then the sequence's bounds with the partials (which do not depend on
// them; rows past the sequence are dropped at the store).
template <int G>
__global__ __launch_bounds__(kMergeThreads) __attribute__((amdgpu_waves_per_eu(1, 4))) void prefill_merge_kernel(
    const AttnArgs a) {
  constexpr int D = kHeadDim;
  constexpr int TM = kPrefillRows / G;
  constexpr int CQ = 8;  // chunks per quarter
  const int r = threadIdx.x;
  const int hkv = a.num_kv_heads;
  // w = (unit, quarter) * hkv + g: with 8 kv heads, head g's merges run on XCD g (work-groups
  // go to XCDs round-robin and the grid is a multiple of 8), where the prefill kernel's
  // sub-queue g wrote its partials, so the reads mostly hit that XCD's L2
  const auto entry = [&](int w) { return a.pf_merges[min((w / hkv) >> 2, a.pf_merge_cap - 1)]; };
  int w = blockIdx.x;
  int4 e = entry(w);
  const int merges = a.pf_queue[kPrefillQueueMeta + 1];
  // the entry is consumed here, so its load goes out with the count's, not after the loop test
  asm volatile("" ::"v"(e.x), "v"(e.y), "v"(e.z), "v"(e.w));
  const int nw = (int)min((int64_t)merges, (int64_t)a.pf_merge_cap * hkv) * 4;
  for (; w < nw; w += gridDim.x, e = entry(w)) {
    const int rest = w / hkv;
    const int g = w - rest * hkv;
    const int c0 = (rest & 3) * CQ;
    const int b = __builtin_amdgcn_readfirstlane(e.x);  // one entry per work-group
    const int qt = __builtin_amdgcn_readfirstlane(e.y);
    const int pg = __builtin_amdgcn_readfirstlane(e.z);
    const int n = __builtin_amdgcn_readfirstlane(e.w);
    if (b < 0 || b >= a.num_seqs || pg < 0 || n <= 0) continue;  // see prefill_item
    if ((int64_t)(pg + n) * hkv > a.pf_part_cap) continue;       // the plan bounds partial ids
    const int q0 = a.cu_q[b];
    const int q1 = a.cu_q[b + 1];
    const int tok = qt * TM + r % TM;
    const int h = g * G + r / TM;
    // Every load below reads a valid split (index clamped to the last one) and a split past
    // the end gets weight 0 by arithmetic on the loaded values (max - inf, sum x 0), which
    // keeps every load unconditional: no load sits behind a branch, so the compiler's wait
    // counts see a whole batch in flight instead of waiting out each load in turn.
    const int last = n - 1;
    const float* ml_base = a.pf_part_ml + ((int64_t)(pg * hkv + g) * kPrefillRows + r) * 2;
    const int64_t ml_step = (int64_t)hkv * kPrefillRows * 2;  // next split of the unit
    const auto load_ml = [&](int s2) {
      const float2 v = *reinterpret_cast<const float2*>(ml_base + min(s2, last) * ml_step);
      return make_float2(v.x + (s2 < n ? 0.f : -INFINITY), v.y * (s2 < n ? 1.f : 0.f));
    };
    const int64_t po_step = (int64_t)hkv * (32 * kPrefillRows * 4);
    const uint16_t* po_base = a.pf_part_o + (int64_t)(pg * hkv + g) * (32 * kPrefillRows * 4) +
                              ((int64_t)c0 * kPrefillRows + r) * 4;
    const auto load = [&](int s2, uint2 (&v)[CQ]) {
#pragma unroll
      for (int c = 0; c < CQ; ++c)
        v[c] = *reinterpret_cast<const uint2*>(po_base + min(s2, last) * po_step + (int64_t)c * kPrefillRows * 4);
    };
    float2 ml[kMergeBatch];
#pragma unroll
    for (int s2 = 0; s2 < kMergeBatch; ++s2) ml[s2] = load_ml(s2);
    uint2 v[kMergeLoads][CQ];
#pragma unroll
    for (int j = 0; j < kMergeLoads; ++j) load(j, v[j]);
    float M = -INFINITY;
#pragma unroll
    for (int s2 = 0; s2 < kMergeBatch; ++s2) M = fmaxf(M, ml[s2].x);
    for (int s2 = kMergeBatch; s2 < n; ++s2) M = fmaxf(M, ml_base[s2 * ml_step]);
    float4 acc[CQ];
#pragma unroll
    for (int c = 0; c < CQ; ++c) acc[c] = make_float4(0.f, 0.f, 0.f, 0.f);
    float L = 0.f;
    // weight 0 for a split past the end or that saw no key (and for every split of a row that
    // saw none: M = -inf)
    const auto add = [&](float2 m, const uint2 (&vv)[CQ]) {
      const float wgt = M == -INFINITY ? 0.f : exp2_fast(m.x - M) * m.y;
      L += wgt;
#pragma unroll
      for (int c = 0; c < CQ; ++c) {
        acc[c].x += wgt * bf16_lo(vv[c].x);
        acc[c].y += wgt * bf16_hi(vv[c].x);
        acc[c].z += wgt * bf16_lo(vv[c].y);
        acc[c].w += wgt * bf16_hi(vv[c].y);
      }
    };
#pragma unroll
    for (int j = 0; j < kMergeLoads; ++j) add(ml[j], v[j]);
    for (int s0 = kMergeLoads; s0 < n; s0 += kMergeLoads) {  // units of many splits
#pragma unroll
      for (int j = 0; j < kMergeLoads; ++j) load(s0 + j, v[j]);
#pragma unroll
      for (int j = 0; j < kMergeLoads; ++j) add(load_ml(s0 + j), v[j]);
    }
    if (tok >= q1 - q0) continue;  // row past the sequence
    const float inv = L > 0.f ? 1.f / L : 0.f;
    uint16_t* op = a.out + (int64_t)(q0 + tok) * a.out_row_stride + h * D + 4 * c0;
#pragma unroll
    for (int c = 0; c < CQ; ++c) {
      uint2 wv;
      wv.x = pack_bf16x2(acc[c].x * inv, acc[c].y * inv);
      wv.y = pack_bf16x2(acc[c].z * inv, acc[c].w * inv);
      *reinterpret_cast<uint2*>(op + 4 * c) = wv;
    }
  }
  // The decode rows' combines (their partials were left by this call's decode launch, which
  // runs first): one (sequence, head) per 128 threads, continuing the work-group order after
  // the split-unit merges so the groups with fewer of those start on these.
  if (a.combine_in_merge) {
    const int pairs = a.num_seqs * a.num_heads;
    const int half = (int)(threadIdx.x >> 7);
    const int grid = (int)gridDim.x;
    const int first = (int)((blockIdx.x + grid - nw % grid) % grid);
    for (int pr = 2 * first + half; pr < pairs; pr += 2 * grid) {
      const int b = pr / a.num_heads;
      combine_row(a, b, pr - b * a.num_heads, threadIdx.x & (kCombineThreads - 1));
    }
  }
}

// ---- Shared-prefix decode ------------------------------------------------------------------
// Decode rows (one query row per sequence) over keys [0, Pb), Pb = min(prefix_keys, Lk), in
// chunks of prefix_chunk keys (one or two whole cache blocks). Work-group (chunk c, kv head g,
// z) serves window z / R of MC = kPrefillRows / G consecutive sequences, as replica z % R. The
// window's sequences whose block tables name the same blocks for the chunk, and that hold the
// same number of keys in it, form a group -- with prefix caching, the sequences sharing those
// blocks; replica r takes the window's groups r, r + R, ... A group's query rows (members x
// the G heads of g) form one MFMA tile set, so each shared block is read once per window
// instead of once per sequence. Every row gets the chunk's (max, sum, numerator) partial in
// the chunk's slot of its sequence, merged with the sequence's split partials by the decode
// combine. A row's arithmetic does not depend on which other rows share its tiles, so results
// do not depend on the grouping (shared or duplicated blocks give identical bits) nor on the
// order of the members inside a group.
//
// The grouping runs in each work-group, on its own window (no plan launch, no plan in memory):
// thread t < MC holds sequence s0 + t's key (keys held in the chunk, its block ids), inserts it
// into an LDS hash table and counts itself into its entry; a group's lead is its lowest
// sequence (an atomic minimum: the same in every replica), and the groups are numbered by their
// leads in sequence order, so all replicas of a window see the same group list. Member ranks
// come from an atomic counter; they only place the rows inside the work-group's own tiles.
template <int G>
__device__ __forceinline__ void shared_prefix_work(const AttnArgs& a, const int c, const int g, const int z) {
  static_assert(kRowBlocks == 1, "one 32-row block per wavefront");
  constexpr int D = kHeadDim;
  constexpr int MC = kPrefillRows / G;  // sequences per window (and rows of one head per tile set)
  constexpr int kHash = 2 * MC;         // hash entries: more than keys, so probing ends
  static_assert(MC <= kPrefillThreads, "one thread per window sequence");
  __shared__ __attribute__((aligned(1024))) char sK[2][kTileBytes];
  __shared__ __attribute__((aligned(1024))) char sV[2][kTileBytes];
  __shared__ int4 s_key[MC];   // (keys held in the chunk, block id, second block id or -1, query row)
  __shared__ int s_owner[kHash], s_lead[kHash], s_size[kHash];
  __shared__ int2 s_group[MC];  // group k: (lead, members)
  __shared__ int s_wave_leads[kPrefillWaves];
  __shared__ int2 s_mem[MC];    // (sequence, query row) of the current group's members
  lds_char* KS[2] = {(lds_char*)sK[0], (lds_char*)sK[1]};
  lds_char* VS[2] = {(lds_char*)sV[0], (lds_char*)sV[1]};

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int BS = a.block_size;
  const int CK = a.prefix_chunk;
  const int Cb = CK / BS;
  const int S = a.num_seqs;
  // work-group (chunk c, kv head g, z = window x replicas + replica)
  const int nrep = a.sp_replicas;
  const int win = z / nrep;
  const int rep = z - win * nrep;
  const int s0 = win * MC;
  const int nwin = min(MC, S - s0);

  // the window's bounds and block-table entries for the chunk in one round of loads (the
  // entries, clamped into the table row, are used only for a sequence holding keys in the
  // chunk, whose entries are valid)
  int4 key = make_int4(0, -1, -1, 0);
  if (tid < nwin) {
    const int b = s0 + tid;
    const int32_t* bt = a.block_table + (int64_t)b * a.bt_stride;
    const int q0 = a.cu_q[b], q1 = a.cu_q[b + 1];
    const int k_lo = a.cu_k[b], k_hi = a.cu_k[b + 1];
    const int id0 = bt[min(c * Cb, a.bt_stride - 1)];
    const int id1 = Cb > 1 ? bt[min(c * Cb + 1, a.bt_stride - 1)] : -1;
    const int Lk = min(k_hi - k_lo, a.max_seqlen_k);
    const int cnt = q1 - q0 == 1 ? max(0, min(CK, min(a.prefix_keys, Lk) - c * CK)) : 0;  // decode rows only
    if (cnt > 0) key = make_int4(cnt, id0, cnt > BS ? id1 : -1, q0);
  }
  if (tid < MC) s_key[tid] = key;
  for (int e = tid; e < kHash; e += kPrefillThreads) {
    s_owner[e] = -1;
    s_lead[e] = MC;
    s_size[e] = 0;
  }
  __syncthreads();
  int slot = -1, rank = 0;
  if (key.x > 0) {
    int h = (int)(((uint32_t)key.y * 2654435761u + (uint32_t)key.z * 40503u) >> 16) & (kHash - 1);
    for (int probe = 0; probe < kHash; ++probe, h = (h + 1) & (kHash - 1)) {
      const int e = atomicCAS(&s_owner[h], -1, tid);
      const int4 k2 = e == -1 ? key : s_key[e];
      if (k2.x == key.x && k2.y == key.y && k2.z == key.z) {
        slot = h;
        break;
      }
    }
    if (slot >= 0) {
      atomicMin(&s_lead[slot], tid);
      rank = atomicAdd(&s_size[slot], 1);
    }
  }
  __syncthreads();
  const int my_lead = slot >= 0 ? s_lead[slot] : -1;
  // group number of a lead: leads below it, in sequence order (ballots per wavefront)
  const bool is_lead = my_lead == tid;
  const uint64_t lead_bits = __builtin_amdgcn_ballot_w64(is_lead);
  if (lane == 0) s_wave_leads[wave] = __builtin_popcountll(lead_bits);
  __syncthreads();
  int before = __builtin_popcountll(lead_bits & ((1ull << lane) - 1ull)), ngroups = 0;
#pragma unroll
  for (int w = 0; w < kPrefillWaves; ++w) {
    const int n = s_wave_leads[w];
    before += w < wave ? n : 0;
    ngroups += n;
  }
  if (is_lead) s_group[before] = make_int2(tid, s_size[slot]);
  __syncthreads();

  const TileLanes tl = tile_lanes(lane);
  const int col = lane & 31;
  const int half = lane >> 5;

  for (int k = rep; k < ngroups; k += nrep) {
    const int2 grp = s_group[k];
    const int4 gkey = s_key[grp.x];
    const int nmem = grp.y;
    const int cnt = gkey.x;
    const int id0 = gkey.y, id1 = gkey.z >= 0 ? gkey.z : gkey.y;
    // tile n: keys 64 n .. of the chunk, in its block (64 n) / BS; rows past cnt re-read the
    // chunk's last key (same block) and are masked
    const auto load = [&](int n, KvRegs& R) {
      const int t0 = n * kTileKeys;
      const int id = t0 < BS ? id0 : id1;
      const int off = t0 % BS;
      const uint16_t* kbase = a.k + (int64_t)id * a.k_block_stride + (int64_t)off * a.k_row_stride + g * D;
      const uint16_t* vbase = a.v + (int64_t)id * a.v_block_stride + (int64_t)off * a.v_row_stride + g * D;
      load_rows(kbase, vbase, load_lanes(a, wave, lane, min(kTileKeys, cnt - 1 - t0)), R);
    };
    // the first two tiles are requested before the members and their q rows (which depend
    // on the member list), so the three rounds of loads overlap
    const int ntiles = (cnt + kTileKeys - 1) / kTileKeys;
    KvRegs R0, R;
    load(0, R0);
    if (ntiles > 1) load(1, R);
    // LDS-only barriers: __syncthreads() would also wait for the tile loads just issued
    lds_barrier();  // s_mem of the previous group has been read
    if (my_lead == grp.x) s_mem[rank] = make_int2(s0 + tid, key.w);
    lds_barrier();

    // rows: 32 per wavefront; TMd = members rounded up to 32 rows per head, head i = row / TMd
    const int TMd = (nmem + 31) & ~31;
    const bool active = wave * 32 < G * TMd;
    const int r0 = wave * 32;
    const int hi = active ? r0 / TMd : 0;
    const int mem = active ? r0 % TMd + col : 0;
    const int2 sm = s_mem[min(mem, nmem - 1)];  // rows past the members read the last one's q
    const int seq = min(max(sm.x, 0), a.num_seqs - 1);
    const int h = g * G + hi;
    bf16x8 qb[kRowBlocks][D / 16];
    {
      const uint16_t* qp = a.q + (int64_t)max(sm.y, 0) * a.q_row_stride + h * D + 8 * half;
#pragma unroll
      for (int kb = 0; kb < D / 16; ++kb)
        qb[0][kb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp + kb * 16));
    }
    f32x16 o[kRowBlocks][4];
    float m_i[kRowBlocks] = {-INFINITY}, l_i[kRowBlocks] = {0.f};
    const int lim[kRowBlocks] = {cnt - 1};  // every member holds the chunk's cnt keys
#pragma unroll
    for (int md = 0; md < 4; ++md)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) o[0][md][rr] = 0.f;

    store_tile_lds(R0, KS[0], VS[0], wave, lane);
    lds_barrier();
    for (int n0 = 0; n0 < ntiles; n0 += 2) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const int n = n0 + st;
        if (n >= ntiles) break;
        const int t0 = n * kTileKeys;
        KvRegs Rn;
        if (n + 2 < ntiles) load(n + 2, Rn);
        const bool full[kRowBlocks] = {t0 + kTileKeys - 1 <= lim[0]};
        if (active) compute_tile(KS[st], VS[st], tl, qb, o, m_i, l_i, t0, lim, full, a.scale_log2, lane);
        if (n + 1 < ntiles) store_tile_lds(R, KS[st ^ 1], VS[st ^ 1], wave, lane);
        lds_barrier();
        R = Rn;
      }
    }

    // partial of (member, head h) for chunk c, in the decode kernel's layout: the normalised
    // output o / l in bf16 and (max, sum); O^T element rr of d-block md is
    // d = 32 md + 8 (rr >> 2) + 4 half + (rr & 3), i.e. four consecutive elements
    const float l_tot = swap_halves_sum(l_i[0]);
    if (active && mem < nmem) {
      const int64_t unit = ((int64_t)seq * a.prefix_stride + c) * a.num_heads + h;
      uint16_t* po = a.part_o + unit * D + 4 * half;
      const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
#pragma unroll
      for (int md = 0; md < 4; ++md)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint2 w;
          w.x = pack_bf16x2(o[0][md][4 * q] * inv, o[0][md][4 * q + 1] * inv);
          w.y = pack_bf16x2(o[0][md][4 * q + 2] * inv, o[0][md][4 * q + 3] * inv);
          *reinterpret_cast<uint2*>(po + 32 * md + 8 * q) = w;
        }
      if (half == 0) *reinterpret_cast<float2*>(a.part_ml + unit * 2) = make_float2(m_i[0], l_tot);
    }
  }
}

// grid (chunk, kv head, window x replicas): work-groups go to the XCDs round-robin by linear
// id, so with z slowest the first replica of every (chunk, head) spreads over all of them
template <int G>
__global__ __launch_bounds__(kPrefillThreads, kWavesPerSimd) void shared_prefix_kernel(const AttnArgs a) {
  shared_prefix_work<G>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// The shared-prefix work and the flat decode grid over the keys after the prefix in one
// launch. Run back to back, the prefix kernel -- a chain of dependent steps in a few dozen
// work-groups (bounds, grouping, member list, q rows, tiles, partials), most of the GPU idle
// -- and the flat grid, which streams the suffixes on every CU, add up; here the first
// sp_groups work-groups take the prefix work (one replica per window) and then sp_tail flat
// groups each, and the sp_decode work-groups after them sp_per flat groups each, as many as
// the CUs left beside the prefix work hold at once. The two kinds write disjoint partial slots
// (prefix chunks, then the flat pieces), merged by the combine pass as before. A work-group's
// eight wavefronts take its flat groups sp_quads at a time (one flat group = the kv heads of
// sp_quads wavefronts); the flat grid's groups are numbered across the work-groups.
template <int G, int U, int R>
__global__ __launch_bounds__(kPrefillThreads, kWavesPerSimd) void shared_prefix_flat_kernel(const AttnArgs a) {
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int blk = blockIdx.x;
  int first, count;  // this work-group's flat groups
  if (blk < a.sp_groups) {
    const int c = blk % a.prefix_slots;
    const int rest = blk / a.prefix_slots;
    shared_prefix_work<G>(a, c, rest % a.num_kv_heads, rest / a.num_kv_heads);
    first = a.sp_decode * a.sp_per + blk * a.sp_tail;
    count = a.sp_tail;
  } else {
    first = (blk - a.sp_groups) * a.sp_per;
    count = a.sp_per;
  }
  const int j = wave / a.sp_quads;  // this wavefront's flat group, and its kv-head quad in it
  const int qd = wave - j * a.sp_quads;
  const int u = first + j;
  if (j < count && u <= a.flat_groups + a.num_seqs)
    flat_decode_piece<G, U, R, true, false, true>(a, u, qd * (4 / R), lane, qd == 0);
}


int device_prefill_slots() {
  static int cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return kPrefillSlotsMax;
  if (cached[dev] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = kPrefillSlotsMax;
    cached[dev] = std::min(cus, kPrefillSlotsMax);  // one work-group per CU
  }
  return cached[dev];
}

// Which kernel a call takes, from its launch bounds (the lengths are on the device): an estimate of the
// key tiles per work-group, with all `rows` prefill rows in sequences of the longest key count's half --
// what the causal limit leaves of fresh rows, and half of the longest cached prefix for the others. The
// w8 kernel starts an item sooner, prefill_kernel's tile takes less. Whole calls with `real` tiles per
// work-group, time of w8 / time of prefill_kernel, with warm caches and with 512 MiB read before each
// call (which evicts the kernels' code too):
//   uniform paged chunks   real 5 0.92 / 0.90   9 0.93 / 0.92   18 0.96 / 0.95   33 1.00 / 0.97
//                          36 1.02 / 1.02   41 1.03 / 1.02   63 1.01 / 1.02   73 1.05 / 1.03
//                          129 1.09 / 1.08   274 1.11 / 1.11
//   uniform fresh prompts  real 9 0.95 / 0.94   18 0.97 / 0.96   33 1.02 / 1.01   36 1.06 / 1.09   68 1.06 / 1.05
//   ragged                 prompts of 100-1024 28 0.97 / 0.97, 34 1.00 / 0.99; of 100-512 21 0.95 / 0.94;
//                          chunks of 512 over 0-4096 keys 24 0.96 / 0.96; of 128-1024 over 1024 38 1.06 / 1.06
// so the line is near 34 real tiles. Fresh prompts of many lengths (flat K/V: their mean is known) count
// with the middle of the mean and the longest, where the longest alone came out a fifth above their
// tiles (31 prompts of 100-1024 took prefill_kernel: 151.7 us, w8 150.0, with the store); chunks that all
// have the longest prefix come out below theirs (half at worst, which leaves up to 3% where they lie
// between 36 and 72).
constexpr int kSmallTiles = 36;
//
// Prefill rows: the call's rows less one per sequence, plus one for each that can be a prefill sequence
// of the longest length. (With every sequence at that length 128 decode rows beside 8 chunks of 100 over
// 2048 keys took prefill_kernel: 182.1 / 192.4 us warm / cold, w8 175.9 / 180.3; beside one chunk of 64
// over 4096 159.2 / 166.2, w8 156.3 / 161.3.)
int64_t prefill_rows_of(int num_seqs, int max_seqlen_q, int64_t num_rows) {
  if (num_rows <= 0) return (int64_t)num_seqs * max_seqlen_q;
  const int64_t more = std::max<int64_t>(num_rows - num_seqs, 0);
  return more + std::min<int64_t>(num_seqs, (more + max_seqlen_q - 2) / (max_seqlen_q - 1));
}

template <int G>
bool small_prefill(const AttnArgs& a, bool paged, bool causal, int max_seqlen_q, int64_t num_rows) {
  constexpr int TM = kPrefillRows / G;
  const int64_t rows = prefill_rows_of(a.num_seqs, max_seqlen_q, num_rows);
  double keys = a.max_seqlen_k;
  if (!paged && num_rows > 0) keys = 0.5 * (keys + std::min(keys, (double)num_rows / a.num_seqs));
  if (causal) keys = 0.5 * (keys + TM);
  return (double)rows * a.num_kv_heads * keys < (double)kSmallTiles * a.pf_slots * TM * kTileKeys;
}

template <int G, bool PAGED, bool CAUSAL>
hipError_t launch_prefill_gpc(const AttnArgs& a, bool small, hipStream_t stream) {
  if (small) {
    hipLaunchKernelGGL((prefill_plan_kernel<G, CAUSAL, true>), dim3(1), dim3(kPlanThreads), 0, stream, a);
    hipLaunchKernelGGL((prefill_w8_kernel<G, PAGED, CAUSAL>), dim3(a.pf_slots), dim3(kPrefillThreads), 0, stream, a);
  } else {
    hipLaunchKernelGGL((prefill_plan_kernel<G, CAUSAL, false>), dim3(1), dim3(kPlanThreads), 0, stream, a);
    hipLaunchKernelGGL((prefill_kernel<G, PAGED, CAUSAL>), dim3(a.pf_slots), dim3(kPfThreads), 0, stream, a);
  }
  hipLaunchKernelGGL((prefill_merge_kernel<G>), dim3(kMergeGroups), dim3(kMergeThreads), 0, stream, a);
  return hipGetLastError();
}

template <int G>
hipError_t launch_prefill_g(const AttnArgs& a, bool paged, bool causal, int max_seqlen_q, int64_t num_rows,
                            hipStream_t stream) {
  constexpr int TM = kPrefillRows / G;
  AttnArgs pa = a;
  pa.prefill_qtiles = (max_seqlen_q + TM - 1) / TM;
  pa.pf_slots = device_prefill_slots();
  pa.flat_step = decode_flat_step(G, a.num_kv_heads);  // the decode pieces' step, for the merge kernel's combines
  const bool small = small_prefill<G>(pa, paged, causal, max_seqlen_q, num_rows);
  if (paged)
    return causal ? launch_prefill_gpc<G, true, true>(pa, small, stream) : launch_prefill_gpc<G, true, false>(pa, small, stream);
  return causal ? launch_prefill_gpc<G, false, true>(pa, small, stream) : launch_prefill_gpc<G, false, false>(pa, small, stream);
}

}  // namespace

template <int G>
void launch_shared_prefix_g(AttnArgs a, hipStream_t stream) {
  // grid (chunk, kv head, window x replicas): windows of kPrefillRows / G sequences, and
  // replicas taking a window's groups in turn, as many as keep the grid near two work-groups
  // per CU (a window usually holds one group per chunk; the spare replicas exit after the
  // grouping)
  constexpr int MC = kPrefillRows / G;
  const int windows = (a.num_seqs + MC - 1) / MC;
  const int pool = 2 * device_prefill_slots();
  a.sp_replicas = std::max(1, std::min(MC, pool / std::max(1, a.prefix_slots * a.num_kv_heads * windows)));
  hipLaunchKernelGGL(shared_prefix_kernel<G>,
                     dim3((unsigned)a.prefix_slots, (unsigned)a.num_kv_heads, (unsigned)(windows * a.sp_replicas)),
                     dim3(kPrefillThreads), 0, stream, a);
}

template <int G, int U, int R>
void launch_shared_prefix_flat_g(const AttnArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((shared_prefix_flat_kernel<G, U, R>), dim3((unsigned)(a.sp_groups + a.sp_decode)),
                     dim3(kPrefillThreads), 0, stream, a);
}

template <int G>
void launch_shared_prefix_flat_gr(const AttnArgs& a, hipStream_t stream) {
  constexpr int U = decode_step_keys(G);
  switch (decode_key_rows(a.num_kv_heads)) {
    case 4: launch_shared_prefix_flat_g<G, U, 4>(a, stream); break;
    case 2: launch_shared_prefix_flat_g<G, U, 2>(a, stream); break;
    default: launch_shared_prefix_flat_g<G, U, 1>(a, stream); break;
  }
}

bool launch_shared_prefix_flat(AttnArgs& a, int group, hipStream_t stream, hipError_t* err) {
  *err = hipSuccess;
  if (a.num_seqs <= 0 || a.prefix_keys <= 0 || a.prefix_slots <= 0 || a.flat_groups <= 0) return false;
  if (!a.block_table || !a.part_o || !a.part_ml || a.num_seqs > kSharedPrefixMaxSeqs ||
      a.prefix_chunk % a.block_size != 0 || a.prefix_chunk / a.block_size > kSharedPrefixMaxChunkBlocks ||
      a.prefix_slots > kCombineMaxSplits)
    return false;
  const int nh = 4 / decode_key_rows(a.num_kv_heads);           // kv heads per wavefront
  const int quads = (a.num_kv_heads + nh - 1) / nh;              // wavefronts per flat group
  if (kPrefillWaves % quads != 0) return false;
  const int per = kPrefillWaves / quads;                         // flat groups per work-group
  const int MC = kPrefillRows / group;
  const int windows = (a.num_seqs + MC - 1) / MC;
  const int64_t P = (int64_t)a.prefix_slots * a.num_kv_heads * windows;
  const int cus = device_prefill_slots();                        // one work-group per CU
  if (P >= cus / 2) return false;                                // little room left for the suffixes
  // decode work-groups fill the CUs beside the prefix ones; those take half a share after
  // their prefix work. The flat grid shrinks to the groups these hold (never grows: the
  // workspace's partial slots are sized for the flat plan's grid).
#ifndef PK_SP_TAIL_DIV
#define PK_SP_TAIL_DIV 2
#endif
  const int tail = PK_SP_TAIL_DIV > 0 ? per / PK_SP_TAIL_DIV : 0;
  const int D = cus - (int)P;
  const int64_t total = (int64_t)D * per + P * tail;             // flat groups, recorder included
  const int W = (int)std::min<int64_t>(a.flat_groups, total - a.num_seqs - 1);
  if (W < 2) return false;
  a.flat_groups = W;
  a.sp_replicas = 1;
  a.sp_groups = (int)P;
  a.sp_decode = D;
  a.sp_per = per;
  a.sp_tail = tail;
  a.sp_quads = quads;
  a.flat_step = decode_flat_step(group, a.num_kv_heads);
  // the decode launch's partial-store policy (kStoreThroughBytes), on this grid's units
  a.store_through = ((int64_t)a.num_seqs + a.flat_groups) * a.num_heads * kHeadDim * 4 > kStoreThroughBytes;
  switch (group) {
    case 1: launch_shared_prefix_flat_gr<1>(a, stream); break;
    case 2: launch_shared_prefix_flat_gr<2>(a, stream); break;
    case 4: launch_shared_prefix_flat_gr<4>(a, stream); break;
    case 8: launch_shared_prefix_flat_gr<8>(a, stream); break;
    default: *err = hipErrorInvalidValue; return true;
  }
  *err = hipGetLastError();
  return true;
}

hipError_t launch_shared_prefix(const AttnArgs& a, int group, hipStream_t stream) {
  if (a.num_seqs <= 0 || a.prefix_keys <= 0 || a.prefix_slots <= 0) return hipSuccess;
  if (!a.block_table || !a.part_o || !a.part_ml || a.num_seqs > kSharedPrefixMaxSeqs ||
      a.prefix_chunk % a.block_size != 0 || a.prefix_chunk / a.block_size > kSharedPrefixMaxChunkBlocks ||
      a.prefix_slots > kCombineMaxSplits)
    return hipErrorInvalidValue;
  switch (group) {
    case 1: launch_shared_prefix_g<1>(a, stream); break;
    case 2: launch_shared_prefix_g<2>(a, stream); break;
    case 4: launch_shared_prefix_g<4>(a, stream); break;
    case 8: launch_shared_prefix_g<8>(a, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_prefill(const AttnArgs& a, int group, bool paged, bool causal, int max_seqlen_q,
                          int64_t num_rows, hipStream_t stream) {
  if (a.num_seqs <= 0 || max_seqlen_q <= 1) return hipSuccess;
  if (!a.pf_queue || !a.pf_items || !a.pf_merges || !a.pf_part_o || !a.pf_part_ml) return hipErrorInvalidValue;
  switch (group) {
    case 1: return launch_prefill_g<1>(a, paged, causal, max_seqlen_q, num_rows, stream);
    case 2: return launch_prefill_g<2>(a, paged, causal, max_seqlen_q, num_rows, stream);
    case 4: return launch_prefill_g<4>(a, paged, causal, max_seqlen_q, num_rows, stream);
    case 8: return launch_prefill_g<8>(a, paged, causal, max_seqlen_q, num_rows, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pk
