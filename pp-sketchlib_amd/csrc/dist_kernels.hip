// HIP kernels for the core/accessory distance path on gfx950 (MI355X).
//
// Hot loop (reference semantics: calc_intersize, dist/dist.cpp:50-78): for a
// pair of samples and one k-mer length, the match count is
//   sum over 64-bin words w of popcount( AND_l NOT(a[w][l] XOR b[w][l]) )
// over the 14 bit layers l.  Here every 64-bit layer word is processed as two
// 32-bit planes; per plane and pair that is one v_xnor_b32 (first layer) plus
// 13 v_bitop3_b32 (acc & ~(a ^ b)) and one v_bcnt_u32_b32: 30 int32 VALU ops
// per 64-bin word per pair, which is the algorithmic op count.
//
// Tiling (GEMM-shaped, integer VALU, no MFMA):
//  * a workgroup owns a tile of pairs for ONE k-mer length: its 8 waves form
//    a grid of row groups x column groups, each wave RQ rows x 64 RR columns
//    (RR columns per lane);
//  * the RQ row samples of a wave are wave-uniform, so their planes are read
//    with scalar loads into SGPRs: each v_bitop3 takes its row operand from
//    an SGPR;
//  * column planes are staged per group of words straight from global memory
//    into LDS (global_load_lds_dwordx4, double buffered) and read per lane;
//  * per-pair counts live in VGPRs for the whole word loop, then go to a
//    per-tile count scratch;
//  * the last of the n_k workgroups of a tile to finish (device-scope atomic)
//    runs the fused epilogue for the tile: random-match correction, Jaccard,
//    log-Jaccard-vs-k regression, dense output.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <numeric>

#include "bin_fraction.h"
#include "log_jaccard.h"
#include "ppsk_internal.h"

namespace ppsk {

// ---------------------------------------------------------------------------
// Stripe transform: raw reference layout -> stripes.
// raw: [count][n_k][s64 * 14] uint64 (word w, layer l at w*14 + l,
// sketch/sketch.cpp:82-92), samples first .. first+count-1 of the set.
// One workgroup per (kk, stripe block, w): the block's 128 sample records
// of 14 uint64 (112 B each, contiguous in raw) are read with 16-byte loads
// into LDS, then the (kk, block, w) slab of 28 planes x 128 samples is
// written as one contiguous 14 KiB run.  Samples of the block outside
// [first, first + count) are left untouched (an upload in several chunks).
// ---------------------------------------------------------------------------
constexpr int STRIPE_TB = 256;
constexpr int STRIPE_REC = BBITS + 1;  // uint64 per LDS record (one pad word)

__global__ __launch_bounds__(STRIPE_TB) void stripe_kernel(const uint64_t* __restrict__ raw,
                                                           int64_t count, int64_t first,
                                                           int32_t n_k, int32_t s64, int32_t nb,
                                                           uint32_t* __restrict__ stripes) {
  __shared__ uint64_t rec[BLK * STRIPE_REC];
  const int64_t blk = (int64_t)first / BLK + blockIdx.y;
  const int kk = (int)(blockIdx.z);
  for (int w = (int)blockIdx.x; w < s64; w += (int)gridDim.x) {
    // samples of this block in this upload: n in [n0, n1)
    const int64_t n0 = blk * BLK > first ? blk * BLK : first;
    const int64_t n1 = (blk + 1) * BLK < first + count ? (blk + 1) * BLK : first + count;
    // load: 7 uint4 per sample record
    for (int x = threadIdx.x; x < BLK * 7; x += STRIPE_TB) {
      const int lane = x / 7, part = x % 7;
      const int64_t n = blk * BLK + lane;
      if (n >= n0 && n < n1) {
        const uint4* src = reinterpret_cast<const uint4*>(
            raw + (((n - first) * n_k + kk) * (int64_t)s64 + w) * BBITS);
        const uint4 v = src[part];
        uint64_t* d = rec + lane * STRIPE_REC + part * 2;
        d[0] = (uint64_t)v.x | ((uint64_t)v.y << 32);
        d[1] = (uint64_t)v.z | ((uint64_t)v.w << 32);
      }
    }
    __syncthreads();
    uint32_t* dst = stripes + (((int64_t)kk * nb + blk) * s64 + w) * (HL * BLK);
    for (int o = threadIdx.x; o < HL * BLK; o += STRIPE_TB) {
      const int hl = o / BLK, lane = o % BLK;
      const int64_t n = blk * BLK + lane;
      if (n >= n0 && n < n1) {
        const int h = hl / BBITS, l = hl % BBITS;
        const uint64_t v = rec[lane * STRIPE_REC + l];
        dst[o] = h ? (uint32_t)(v >> 32) : (uint32_t)v;
      }
    }
    __syncthreads();
  }
}

hipError_t launch_stripe(const uint64_t* raw, int64_t count, int64_t first,
                         int32_t n_k, int32_t s64, int32_t nb, uint32_t* stripes,
                         hipStream_t stream) {
  if (count <= 0) return hipSuccess;
  const int64_t b0 = first / BLK, b1 = (first + count - 1) / BLK;
  const unsigned words = (unsigned)(s64 < 64 ? s64 : 64);  // grid x strides over words
  dim3 grid(words, (unsigned)(b1 - b0 + 1), (unsigned)n_k);
  stripe_kernel<<<grid, STRIPE_TB, 0, stream>>>(raw, count, first, n_k, s64, nb, stripes);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Helpers
// ---------------------------------------------------------------------------
typedef const __attribute__((address_space(4))) uint32_t CU32;
typedef const __attribute__((address_space(4))) DistParams CParams;
typedef const __attribute__((address_space(4))) CodeGroup CCodeGroup;

__device__ __forceinline__ uint32_t match_and(uint32_t acc, uint32_t a, uint32_t b) {
  // truth table over (acc, a, b) with src0 = 0xF0, src1 = 0xCC, src2 = 0xAA:
  // acc & ~(a ^ b) = 0x90
  return __builtin_amdgcn_bitop3_b32(acc, a, b, 0x90);
}

// v_bcnt_u32_b32 with accumulate: cnt + popcount(x) in one VALU op (the
// compiler otherwise splits paired popcounts into two bcnt and a v_add3).
__device__ __forceinline__ uint32_t bcnt_acc(uint32_t x, uint32_t cnt) {
  uint32_t r;
  asm("v_bcnt_u32_b32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(cnt));
  return r;
}

// Per-pair epilogue pieces.  Reference semantics (CPU path):
//  J_obs = c / (64 * s64)                        reference.cpp:222-232
//  J     = max(J_obs - r, 0) * 1 / (1 - r)       dist/dist.hpp:13-24 (double)
//  dists[kk] = (float) J                         linear_regression.cpp:62-71
//  window [first J > tol, last J > tol], LS of log J on k, core/acc
//                                                linear_regression.cpp:16-60
template <typename P>
__device__ __forceinline__ double random_for(const P& p, int kk, int64_t gi, int64_t gj) {
  if (p.random_mode == RANDOM_EQUAL_BASE) {
    // csrs combination (random_match.cpp:333-334) of per-sample terms
    const double j1 = p.jv_rows[gi * p.n_k + kk];
    const double j2 = p.jv_cols[gj * p.n_k + kk];
    double r = 0.0;
    if (j1 > 0 && j2 > 0) r = (j1 * j2) / (j1 + j2 - j1 * j2);
    return r;
  }
  if (p.random_mode == RANDOM_MC) {
    const int C = p.n_clusters;
    const int cr = p.cl_rows[gi], cc = p.cl_cols[gj];
    const int a = p.mc_ref_is_col ? cc : cr;
    const int b = p.mc_ref_is_col ? cr : cc;
    return (double)p.mc_table[(kk * C + a) * C + b];
  }
  return 0.0;
}

// Cancellation request of the call (ppsk_cancel), read from host-mapped
// memory with a system-scope load so that no cache holds a stale value.
__device__ __forceinline__ bool cancel_seen(const uint32_t* flag) {
  return flag != nullptr &&
         __hip_atomic_load(const_cast<uint32_t*>(flag), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM) != 0u;
}

// n more (tile, k-mer length) items finished: the device counter, mirrored
// into the host-mapped progress word with a plain store.
__device__ __forceinline__ void add_progress(const Control& c, unsigned long long n) {
  if (c.progress == nullptr) return;
  const unsigned long long old = atomicAdd(c.progress, n);
  if (c.progress_host != nullptr) {
    __hip_atomic_store(c.progress_host, old + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Whether the call of an item of a split pass was cancelled (one lane of workgroup
// `block` asks).  The host's flag and the mirrored progress cross one link for all
// CUs, about 0.1 us each: read and written in every item, 4,400 short items took
// 863 us instead of 433.  So one item in 64 reads the flag and passes it on in a
// device word that the others read, and one in 64 mirrors the progress.  The
// first workgroups of a call, which start together right after the host has
// looked, read neither; nor does a pass of less than about 2 ms, which ends
// before a request could stop it (its call reports the request and the final
// count all the same): looking took 37 of the 223 us of one query against 6,000.
constexpr uint32_t ITEM_WATCH = 64, ITEM_MIRROR = 64;

__device__ __forceinline__ bool item_stopped(const Control& c, uint32_t block) {
  if (__hip_atomic_load(c.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return true;
  if (block % ITEM_WATCH != 0 || !cancel_seen(c.cancel)) return false;
  __hip_atomic_store(c.stop, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

__device__ __forceinline__ void add_item(const Control& c) {
  if (c.progress == nullptr) return;
  const unsigned long long done = atomicAdd(c.progress, 1ull) + 1ull;
  if (c.progress_host != nullptr && done % ITEM_MIRROR == 0) {
    __hip_atomic_store(c.progress_host, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__device__ __forceinline__ double jaccard_d(uint32_t c, double bins, double rbins, double r) {
  const double obs = bin_fraction(c, bins, rbins);
  const double diff = obs > r ? (obs - r) : 0.0;
  return (diff * 1.0) / (1.0 - r);
}

// Table of the regression's logarithm (log_jaccard.h); every device holds a
// copy, written once when the library sets the device up.
__device__ double g_log_tab[LOG_TAB_DOUBLES];


// ---------------------------------------------------------------------------
// Tile shape and LDS staging
// ---------------------------------------------------------------------------
// A stage is WS words x 28 planes x TC dwords = 1792 uint4 (28 KiB), double
// buffered (56 KiB per workgroup, two workgroups per CU).  Stages are copied
// global -> LDS directly: round i of wave w moves uint4 [i*512 + w*64, +64)
// of the stage; the last round is a half round.
//
// The 8 waves form a grid of RG row groups x CG column groups: wave w takes
// rows (w / CG) * RQ .. +RQ and columns (w % CG) * 64 RR .. +64 RR of the
// tile (lane l: columns l + 64 r, r < RR, of its group).  Every column
// operand a lane reads from LDS meets RQ row operands, so the VALU work per
// LDS byte is RQ / 4 ops: at RQ = 8 that matches the CU's VALU issue rate
// (256 lane-ops per clock) to its LDS read rate (128 B per clock).  The
// pipelined shapes therefore all keep RQ = 8 and span 256 columns
// (CG = 4 / RR): 64 x 256 (8 x 1 waves), 32 x 256 (4 x 2), 16 x 256 (2 x 4).
// The compiler-scheduled shapes (RQ = 16) stack all waves on the rows.
template <int RQ, int RR>
struct TileCfg {
  static constexpr int CG = RQ == 8 ? 4 / RR : 1;
  static constexpr int RG = WAVES / CG;
  static constexpr int TROWS = RG * RQ;
  static constexpr int TC = CG * 64 * RR;
  static constexpr int WS = 4 / (CG * RR);
  static_assert(CG * RG == WAVES, "the wave grid covers the workgroup");
  static constexpr int STAGE_U4 = WS * HL * TC / 4;  // 1792
  static constexpr int ROUNDS = (STAGE_U4 + WAVES * 64 - 1) / (WAVES * 64);  // 4
  static_assert(STAGE_U4 % 64 == 0, "stage must be whole wave rounds");
  static_assert(BLK % TROWS == 0, "row tiles must not straddle stripe blocks");
  // row panel of one stage (WS words x 28 planes x TROWS samples) in uint4
  static constexpr int ROW_U4 = WS * HL * TROWS / 4;
  static constexpr int ROW_ROUNDS = (ROW_U4 + WAVES * 64 - 1) / (WAVES * 64);
  // LDS target of the row prefetch: whole waves of uint4 (never read)
  static constexpr int ROW_LDS_U4 = (ROW_U4 + 63) / 64 * 64;
};

// s_waitcnt vmcnt(n) with expcnt / lgkmcnt left unconstrained (gfx9 encoding)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// LDS byte address of a __shared__ object.
__device__ __forceinline__ uint32_t lds_addr(const uint4* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// One 16-byte-per-lane global -> LDS copy: lane L reads saddr + voff (bytes)
// and writes LDS bytes [lds_base + OFF + 16 L, +16).  Written as inline asm
// so that the compiler's wait-count pass does not treat it as a pending write
// to every LDS buffer (it cannot tell the two stage buffers apart and would
// wait for the copy of the next stage before reading the current one);
// completion is awaited explicitly with vmcnt before the stage barrier.  The
// LDS address is base + OFF with OFF an immediate, so a stage needs one SGPR
// per buffer rather than one per copy.
template <int OFF>
__device__ __forceinline__ void dma16(const uint32_t* saddr, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_add_u32 m0, %0, %3\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_base), "v"(voff), "s"(saddr), "i"(OFF)
               : "memory", "m0", "scc");
}

// Workgroup barrier without the release/acquire fences of __syncthreads():
// those wait for every outstanding vector-memory operation, including the
// next stage's direct-to-LDS copy that is meant to overlap the matching.
// Ordering of the stage copies is handled explicitly with vmcnt waits.
__device__ __forceinline__ void stage_barrier() { asm volatile("s_barrier" ::: "memory"); }

// Column operands of one stage: words [w0, w0 + WS) of the tile's TC columns,
// which may span two stripe blocks (TC = 256) or half of one (TC = 64).
// Columns past the last stripe block read the last block (masked later).
// Round I of wave w copies uint4 [I * 512 + w * 64, +64) of the stage.
//
// Addressing: a lane's source is (tile column base) + (w0 * plane slab) +
// (its byte offset within the tile's <= 2 stripe blocks).  The last term does
// not depend on the word, so it is computed once per tile (ColOffsets, one
// VGPR per round, < 2^32 since it spans at most two blocks of one word group)
// and every stage only moves the scalar base.
template <int RQ, int RR>
struct ColOffsets {
  uint32_t v[TileCfg<RQ, RR>::ROUNDS];
};

template <int RQ, int RR>
__device__ __forceinline__ ColOffsets<RQ, RR> col_offsets(int64_t col0, int nb_cols, int s64,
                                                          int wave, int lane) {
  using Cfg = TileCfg<RQ, RR>;
  constexpr int TC = Cfg::TC;
  ColOffsets<RQ, RR> o;
  const int blk0 = (int)(col0 / BLK);
#pragma unroll
  for (int i = 0; i < Cfg::ROUNDS; ++i) {
    const int x = i * (WAVES * 64) + wave * 64 + lane;
    const int row = x / (TC / 4);  // ws * HL + hl
    const int64_t col = col0 + (x % (TC / 4)) * 4;
    int blk = (int)(col / BLK);
    blk = blk < nb_cols ? blk : nb_cols - 1;
    const uint32_t e = (uint32_t)(blk - blk0) * (uint32_t)s64 * (HL * BLK) +
                       (uint32_t)row * BLK + (uint32_t)(col % BLK);
    o.v[i] = e * 4u;
  }
  return o;
}

template <int RQ, int RR, int I>
__device__ __forceinline__ void issue_round(const uint32_t* sbase, const ColOffsets<RQ, RR>& off,
                                            uint32_t wbase, int wave) {
  using Cfg = TileCfg<RQ, RR>;
  if constexpr (I < Cfg::ROUNDS) {
    if (I * (WAVES * 64) + wave * 64 < Cfg::STAGE_U4) {  // wave-uniform
      dma16<I * WAVES * 64 * 16>(sbase, off.v[I], wbase);
    }
    issue_round<RQ, RR, I + 1>(sbase, off, wbase, wave);
  }
}

// Row-panel prefetch: the stage's row planes (read later with scalar loads)
// are copied into a scratch LDS area one stage ahead, only so that the scalar
// loads find them in L2.  Lane offsets as for the columns.
template <int RQ, int RR>
struct RowOffsets {
  uint32_t v[TileCfg<RQ, RR>::ROW_ROUNDS];
};

template <int RQ, int RR>
__device__ __forceinline__ RowOffsets<RQ, RR> row_offsets(int wave, int lane) {
  using Cfg = TileCfg<RQ, RR>;
  constexpr int PER_PLANE = Cfg::TROWS / 4;  // uint4 per plane of the panel
  RowOffsets<RQ, RR> o;
#pragma unroll
  for (int i = 0; i < Cfg::ROW_ROUNDS; ++i) {
    int x = i * (WAVES * 64) + wave * 64 + lane;
    if (x >= Cfg::ROW_U4) x = 0;  // lanes past the panel repeat its first uint4
    const int plane = x / PER_PLANE;  // ws * HL + hl
    const int part = x % PER_PLANE;
    o.v[i] = (uint32_t)(plane * BLK + part * 4) * 4u;
  }
  return o;
}

template <int RQ, int RR, int I>
__device__ __forceinline__ void prefetch_round(const uint32_t* rbase, const RowOffsets<RQ, RR>& off,
                                               uint32_t wbase, int wave) {
  using Cfg = TileCfg<RQ, RR>;
  if constexpr (I < Cfg::ROW_ROUNDS) {
    if (I * (WAVES * 64) + wave * 64 < Cfg::ROW_U4) {  // wave-uniform
      dma16<I * WAVES * 64 * 16>(rbase, off.v[I], wbase);
    }
    prefetch_round<RQ, RR, I + 1>(rbase, off, wbase, wave);
  }
}

// sbase: the tile's first column block, word w0 (wave-uniform).
template <int RQ, int RR>
__device__ __forceinline__ void issue_stage(const uint32_t* sbase, const ColOffsets<RQ, RR>& off,
                                            uint4* buf, int wave) {
  const uint32_t wbase = lds_addr(buf) + (uint32_t)(wave * 64 * 16);
  issue_round<RQ, RR, 0>(sbase, off, wbase, wave);
}

// ---------------------------------------------------------------------------
// Matching, row operands left to the compiler (PB = 0): one plane at a time.
// ---------------------------------------------------------------------------
template <int RQ, int RR>
__device__ __forceinline__ void match_stage_plain(const CU32* arow, int w0, int nw,
                                                  const uint32_t* sB, int lane,
                                                  uint32_t (&cnt)[RQ][RR]) {
  constexpr int TC = TileCfg<RQ, RR>::TC;
  static_assert(TileCfg<RQ, RR>::CG == 1, "compiler-scheduled shapes stack waves on rows");
  for (int ws = 0; ws < nw; ++ws) {
    const CU32* aw = arow + (int64_t)(w0 + ws) * (HL * BLK);
    const uint32_t* bw = sB + ws * (HL * TC) + lane;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t acc[RQ][RR];
#pragma unroll
      for (int l = 0; l < BBITS; ++l) {
        const int hl = h * BBITS + l;
        uint32_t a[RQ], b[RR];
#pragma unroll
        for (int q = 0; q < RQ; ++q) a[q] = aw[hl * BLK + q];
#pragma unroll
        for (int r = 0; r < RR; ++r) b[r] = bw[hl * TC + 64 * r];
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
#pragma unroll
          for (int r = 0; r < RR; ++r) {
            acc[q][r] = (l == 0) ? ~(a[q] ^ b[r]) : match_and(acc[q][r], a[q], b[r]);
          }
        }
      }
#pragma unroll
      for (int q = 0; q < RQ; ++q)
#pragma unroll
        for (int r = 0; r < RR; ++r) cnt[q][r] = bcnt_acc(acc[q][r], cnt[q][r]);
    }
  }
}

// ---------------------------------------------------------------------------
// Matching with an explicit two-deep operand pipeline (PB = 1 or 2).
// Scalar loads return out of order, so the only possible wait for them is
// "all outstanding" (lgkmcnt(0)), which also covers every LDS read; left to
// itself the compiler issues one plane's s_load and waits for it right away,
// exposing the full L2 latency every RQ * RR VALU ops.  Here the row
// operands of PB planes (scalar loads into SGPR tuples) and the matching
// column operands (ds_read2st64 into VGPR pairs) form one batch: batch b+1
// is issued before batch b is matched, and a single wait that names the
// registers it completes follows the matching.  Each round trip therefore
// overlaps PB * RQ * RR bitop3 of the same wave plus the other waves of the
// SIMD.  All loads of the pipeline are issued from inline asm, so the
// compiler's own wait counting never sees (or waits on) them.
// ---------------------------------------------------------------------------
template <int RQ>
struct ATuple;
template <>
struct ATuple<16> {
  typedef uint32_t T __attribute__((ext_vector_type(16)));
};
template <>
struct ATuple<8> {
  typedef uint32_t T __attribute__((ext_vector_type(8)));
};
template <>
struct ATuple<4> {
  typedef uint32_t T __attribute__((ext_vector_type(4)));
};
template <>
struct ATuple<2> {
  typedef uint32_t T __attribute__((ext_vector_type(2)));
};
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Column operands come in pairs from one ds_read2st64_b32: two column blocks
// of one plane (RR >= 2), or one column of two consecutive planes (RR = 1).
template <int RR, int PB>
struct ColRegs {
  static constexpr int N = RR >= 2 ? PB * (RR / 2) : PB / 2;
};

template <int RQ, int RR, int PB>
struct Batch {
  static_assert(RR >= 2 ? RR % 2 == 0 : PB % 2 == 0, "column operands are read in pairs");
  typename ATuple<RQ>::T a[PB];     // row planes: RQ samples each
  u32x2 b[ColRegs<RR, PB>::N];      // column planes: RR per lane and plane
};

// Column operand (plane pb of the batch, column block r) of a batch.
template <int RQ, int RR, int PB>
__device__ __forceinline__ uint32_t col_operand(const Batch<RQ, RR, PB>& x, int pb, int r) {
  if constexpr (RR >= 2) {
    return x.b[pb * (RR / 2) + r / 2][r % 2];
  } else {
    return x.b[pb / 2][pb % 2];
  }
}

template <int RQ, int OFF>
__device__ __forceinline__ void a_load(const CU32* aw, typename ATuple<RQ>::T& x) {
  if constexpr (RQ == 16) {
    asm volatile("s_load_dwordx16 %0, %1, %2" : "=&s"(x) : "s"(aw), "i"(OFF));
  } else if constexpr (RQ == 8) {
    asm volatile("s_load_dwordx8 %0, %1, %2" : "=&s"(x) : "s"(aw), "i"(OFF));
  } else if constexpr (RQ == 4) {
    asm volatile("s_load_dwordx4 %0, %1, %2" : "=&s"(x) : "s"(aw), "i"(OFF));
  } else {
    static_assert(RQ == 2, "row operands come in SGPR tuples of 2, 4, 8 or 16");
    asm volatile("s_load_dwordx2 %0, %1, %2" : "=&s"(x) : "s"(aw), "i"(OFF));
  }
}

// Issue planes P0 .. P0+PB-1 of the word at (aw, bw); P0 = HL addresses the
// first planes of the next word.  bw is the LDS byte address of plane 0 at the
// lane's first column (a stage holds TC columns per plane); column block r of
// plane P sits at bw + (P TC + 64 r) 4, i.e. at offset P TC / 64 + r in the
// 256-byte units of ds_read2st64.
template <int RQ, int RR, int PB, int P0>
__device__ __forceinline__ void batch_issue(const CU32* aw, uint32_t bw, Batch<RQ, RR, PB>& x) {
  constexpr int TC = TileCfg<RQ, RR>::TC;  // plane stride of the LDS stage
#pragma unroll
  for (int pb = 0; pb < PB; ++pb) {
    if (pb == 0) a_load<RQ, P0 * BLK * 4>(aw, x.a[0]);
    if (pb == 1) a_load<RQ, (P0 + 1) * BLK * 4>(aw, x.a[PB - 1]);
  }
  if constexpr (RR >= 2) {
#pragma unroll
    for (int pb = 0; pb < PB; ++pb) {
#pragma unroll
      for (int rp = 0; rp < RR / 2; ++rp) {
        asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3"
                     : "=&v"(x.b[pb * (RR / 2) + rp])
                     : "v"(bw), "i"((P0 + pb) * TC / 64 + 2 * rp),
                       "i"((P0 + pb) * TC / 64 + 2 * rp + 1));
      }
    }
  } else {
    // one column: planes P0 + pb and P0 + pb + 1 in one read
#pragma unroll
    for (int pb = 0; pb < PB; pb += 2) {
      asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3"
                   : "=&v"(x.b[pb / 2])
                   : "v"(bw), "i"((P0 + pb) * TC / 64), "i"((P0 + pb + 1) * TC / 64));
    }
  }
}

template <int RQ, int RR, int PB>
__device__ __forceinline__ void batch_wait(Batch<RQ, RR, PB>& x) {
  if constexpr (PB == 2 && RR == 4) {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+s"(x.a[0]), "+s"(x.a[1]), "+v"(x.b[0]), "+v"(x.b[1]), "+v"(x.b[2]),
                   "+v"(x.b[3]));
  } else if constexpr (PB == 2 && RR == 2) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(x.a[0]), "+s"(x.a[1]), "+v"(x.b[0]), "+v"(x.b[1]));
  } else if constexpr (PB == 2 && RR == 1) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(x.a[0]), "+s"(x.a[1]), "+v"(x.b[0]));
  } else if constexpr (PB == 1 && RR == 4) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(x.a[0]), "+v"(x.b[0]), "+v"(x.b[1]));
  } else {
    static_assert(PB == 1 && RR == 2, "unsupported batch shape");
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(x.a[0]), "+v"(x.b[0]));
  }
}

// Keeps a batch's registers alive (unchanged) at this point of the program.
// Placed right after the next batch's loads are issued, it stops the
// compiler from matching the current batch first and then reusing its
// registers for the next batch's loads, which would serialise every load
// round trip behind the matching.
template <int RQ, int RR, int PB>
__device__ __forceinline__ void batch_hold(Batch<RQ, RR, PB>& x) {
  if constexpr (PB == 2 && RR == 4) {
    asm volatile("" : "+s"(x.a[0]), "+s"(x.a[1]), "+v"(x.b[0]), "+v"(x.b[1]), "+v"(x.b[2]),
                      "+v"(x.b[3]));
  } else if constexpr (PB == 2 && RR == 2) {
    asm volatile("" : "+s"(x.a[0]), "+s"(x.a[1]), "+v"(x.b[0]), "+v"(x.b[1]));
  } else if constexpr (PB == 2 && RR == 1) {
    asm volatile("" : "+s"(x.a[0]), "+s"(x.a[1]), "+v"(x.b[0]));
  } else if constexpr (PB == 1 && RR == 4) {
    asm volatile("" : "+s"(x.a[0]), "+v"(x.b[0]), "+v"(x.b[1]));
  } else {
    static_assert(PB == 1 && RR == 2, "unsupported batch shape");
    asm volatile("" : "+s"(x.a[0]), "+v"(x.b[0]));
  }
}

// Planes P .. P+PB-1 of one word against the lane's RR columns.
template <int RQ, int RR, int PB, int P>
__device__ __forceinline__ void match_batch(const Batch<RQ, RR, PB>& x, uint32_t (&acc)[RQ][RR]) {
#pragma unroll
  for (int pb = 0; pb < PB; ++pb) {
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        const uint32_t a = x.a[pb][q];
        const uint32_t b = col_operand<RQ, RR, PB>(x, pb, r);
        if ((P + pb) % BBITS == 0) {
          acc[q][r] = ~(a ^ b);
        } else {
          acc[q][r] = match_and(acc[q][r], a, b);
        }
      }
    }
  }
}

// Batches B .. NB-1 of one word; cur holds batch B (loaded and complete).
// The last batch prefetches the first batch of the next word (if any) into
// the registers the next word starts from.
template <int RQ, int RR, int PB, int B>
__device__ __forceinline__ void match_batches(const CU32* aw, uint32_t bw, bool next_word,
                                              Batch<RQ, RR, PB>& cur, Batch<RQ, RR, PB>& nxt,
                                              uint32_t (&acc)[RQ][RR], uint32_t (&cnt)[RQ][RR]) {
  constexpr int NB = HL / PB;
  if constexpr (B + 1 < NB) {
    batch_issue<RQ, RR, PB, (B + 1) * PB>(aw, bw, nxt);
  } else {
    if (next_word) batch_issue<RQ, RR, PB, HL>(aw, bw, nxt);  // word w + 1
  }
  batch_hold<RQ, RR, PB>(cur);
  match_batch<RQ, RR, PB, B * PB>(cur, acc);
  if constexpr (((B + 1) * PB) % BBITS == 0) {
    // end of a 32-bit half: fold its matches into the counts
#pragma unroll
    for (int q = 0; q < RQ; ++q)
#pragma unroll
      for (int r = 0; r < RR; ++r) cnt[q][r] = bcnt_acc(acc[q][r], cnt[q][r]);
  }
  if constexpr (B + 1 < NB) {
    batch_wait<RQ, RR, PB>(nxt);
    match_batches<RQ, RR, PB, B + 1>(aw, bw, next_word, nxt, cur, acc, cnt);
  }
}

// col: the lane's first column within the tile ((wave % CG) * 64 RR + lane).
template <int RQ, int RR, int PB>
__device__ __forceinline__ void match_stage_pipe(const CU32* arow, int w0, int nw,
                                                 const uint4* sbuf, int col,
                                                 uint32_t (&cnt)[RQ][RR]) {
  constexpr int TC = TileCfg<RQ, RR>::TC;
  static_assert((HL / PB) % 2 == 0, "an even batch count keeps the register sets aligned");
  Batch<RQ, RR, PB> c, n;
  const CU32* aw = arow + (int64_t)w0 * (HL * BLK);
  uint32_t bw = lds_addr(sbuf) + col * 4;
  batch_issue<RQ, RR, PB, 0>(aw, bw, c);
  for (int ws = 0; ws < nw; ++ws) {
    batch_wait<RQ, RR, PB>(c);
    uint32_t acc[RQ][RR];
    // batches alternate (c, n); the last one (odd) leaves the next word's
    // first batch in c
    match_batches<RQ, RR, PB, 0>(aw, bw, ws + 1 < nw, c, n, acc, cnt);
    aw += HL * BLK;
    bw += HL * TC * 4;
  }
}

// ---------------------------------------------------------------------------
// Output of one pair (row gi, column gj) from its match counts.  counts(k0, c)
// reads those of k-mer lengths k0 .. k0 + 3 (as far as there are so many) into
// c[0..3]: together, so that a pair waits for memory once per 4 lengths.
// ---------------------------------------------------------------------------
constexpr int OUT_K = 4;

template <typename P>
__device__ __forceinline__ bool pair_valid(const P& p, int64_t gi, int64_t gj) {
  if (p.self_mode && !p.full_square) return gi < gj && gj < p.n_cols;
  return gi < p.n_rows && gj < p.n_cols;
}

template <typename P, typename Counts>
__device__ __forceinline__ void pair_output(const P& p, int64_t gi, int64_t gj, double bins,
                                            double rbins, Counts counts) {
  int64_t pos;
  if (p.full_square) {
    pos = (gi - p.square_row0) * p.out_stride_rows + gj;
  } else if (p.self_mode) {
    pos = p.n_cols * gi - ((gi * (gi + 1)) >> 1) + gj - 1 - gi;  // square_to_condensed
  } else {
    pos = gi * p.n_cols + gj;  // query-major: q * n_ref + r
  }
  pos -= p.out_row_offset;
  const int n_k = p.n_k;
  uint32_t c[OUT_K];
  if (p.out_kind == OUT_COUNTS) {
    uint16_t* o = reinterpret_cast<uint16_t*>(p.out) + pos * n_k;
    for (int k0 = 0; k0 < n_k; k0 += OUT_K) {
      counts(k0, c);
#pragma unroll
      for (int i = 0; i < OUT_K; ++i) {
        if (k0 + i < n_k) o[k0 + i] = (uint16_t)c[i];
      }
    }
    return;
  }
  if (p.out_kind == OUT_JACCARD) {
    float* o = reinterpret_cast<float*>(p.out) + pos * n_k;
    for (int k0 = 0; k0 < n_k; k0 += OUT_K) {
      counts(k0, c);
#pragma unroll
      for (int i = 0; i < OUT_K; ++i) {
        if (k0 + i < n_k) {
          o[k0 + i] = (float)jaccard_d(c[i], bins, rbins, random_for(p, k0 + i, gi, gj));
        }
      }
    }
    return;
  }
  if (p.out_kind == OUT_ONE_MINUS_J) {
    // kNN on Jaccards: (float)(1 - J) of the first two k-mer lengths
    // (src/api.cpp:368-371 narrows 1.0f - double J to float)
    float v[2] = {INFINITY, INFINITY};
    counts(0, c);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k < n_k) {
        v[k] = (float)(1.0 - jaccard_d(c[k], bins, rbins, random_for(p, k, gi, gj)));
      }
    }
    reinterpret_cast<float2*>(p.out)[pos] = make_float2(v[0], v[1]);
    return;
  }
  // core/acc: streaming window fit.  Points before the first valid one are
  // dropped; invalid points after the last valid one are held as pending
  // sums and committed only if a later valid point arrives.
  int first = -1, last = -1;
  double sy = 0.0, sxy = 0.0, py = 0.0, pxy = 0.0;
  for (int k0 = 0; k0 < n_k; k0 += OUT_K) {
    counts(k0, c);
#pragma unroll
    for (int i = 0; i < OUT_K; ++i) {
      const int k = k0 + i;
      if (k >= n_k) break;
      const float jf = (float)jaccard_d(c[i], bins, rbins, random_for(p, k, gi, gj));
      const bool ok = (double)jf > p.tolerance;
      if (!ok && first < 0) continue;
      const double x = (double)p.kvals[k];
      const double y = log_jaccard(jf, g_log_tab);
      if (ok) {
        if (first < 0) {
          first = k;
          sy = y;
          sxy = x * y;
        } else {
          sy += py + y;
          sxy += pxy + x * y;
        }
        py = 0.0;
        pxy = 0.0;
        last = k;
      } else {
        py += y;
        pxy += x * y;
      }
    }
  }
  float core = 0.0f, accd = 0.0f;
  if (first < 0 || last - first + 1 < 2) {
    atomicAdd(p.fail_count, 1ull);
    atomicMin(p.fail_first, (unsigned long long)(pos + p.out_row_offset));
    if (p.fail_rows) atomicAdd(&p.fail_rows[gi], 1u);
  } else {
    const double n = (double)(last - first + 1);
    double sx = 0.0, sxx = 0.0;
    for (int k = first; k <= last; ++k) {
      const double x = (double)p.kvals[k];
      sx += x;
      sxx += x * x;
    }
    const double mx = sx / n;
    const double my = sy / n;
    // centred sums: Sxx = sum x^2 - n mx^2, Sxy = sum xy - n mx my
    const double cxx = sxx - n * mx * mx;
    const double cxy = sxy - n * mx * my;
    const double slope = cxy / cxx;
    const double intercept = my - slope * mx;
    if (slope < 0) core = (float)(1.0 - exp(slope));
    if (intercept < 0) accd = (float)(1.0 - exp(intercept));
  }
  reinterpret_cast<float2*>(p.out)[pos] = make_float2(core, accd);
}

// ---------------------------------------------------------------------------
// Fused epilogue of one tile (run by the last of its n_k workgroups):
// per-k counts -> random-corrected Jaccard -> dense output.  Out of line so
// that none of its state occupies registers during the matching loop.
// ---------------------------------------------------------------------------
// tile_counts: the tile's count block [n_k][tile rows][tile cols].
template <int RQ, int RR>
__device__ __noinline__ void tile_epilogue(CParams* pp, const uint16_t* tile_counts, Tile tile,
                                           int wave, int lane) {
  CParams& p = *pp;
  using Cfg = TileCfg<RQ, RR>;
  constexpr int TC = Cfg::TC;
  constexpr int TROWS = Cfg::TROWS;
  const double bins = 64.0 * (double)p.s64;
  const double rbins = 1.0 / bins;
  // this wave's rows and this lane's first column in the tile (wave grid)
  const int wrow = (wave / Cfg::CG) * RQ;
  const int wcol = (wave % Cfg::CG) * 64 * RR + lane;
  const int64_t gi0 = (int64_t)tile.bi * TROWS + wrow;
  const int64_t col0 = (int64_t)tile.ct * TC + wcol - lane;
  const uint16_t* tbase = tile_counts + (int64_t)wrow * TC + wcol;
  const int64_t kstride = (int64_t)TROWS * TC;
  for (int q = 0; q < RQ; ++q) {
    const int64_t gi = gi0 + q;
    for (int r = 0; r < RR; ++r) {
      const int64_t gj = col0 + lane + 64 * r;
      if (!pair_valid(p, gi, gj)) continue;
      const uint16_t* cp = tbase + q * TC + 64 * r;
      pair_output(p, gi, gj, bins, rbins, [&](int k0, uint32_t (&c)[OUT_K]) {
#pragma unroll
        for (int i = 0; i < OUT_K; ++i) c[i] = cp[min(k0 + i, p.n_k - 1) * kstride];
      });
    }
  }
}

// ---------------------------------------------------------------------------
// Match counts of one tile for k-mer length index kk into cnt (zeroed here).
// pp: the distance parameters, read with scalar loads (kernarg segment or a
// job table entry).  sB0 / sB1: the two LDS stage buffers.
// ---------------------------------------------------------------------------
// The stage loop of tile_match with a narrower matching, for the diagonal
// tiles of a self pass (tile_match_diagonal below).  Copies and the row
// prefetch follow the tile's shape <RQ, RR>; the matching covers MR column
// blocks of 64 per lane from tile column `col`, against the same column
// stage (same plane stride and words per stage).  tile_match keeps its own
// copy of this loop so that the code of the kernels without the diagonal
// path stays exactly as it is.
template <int RQ, int RR, int PB, int MR>
__device__ __forceinline__ void tile_stages(const CU32* arow, const uint32_t* cbase,
                                            const ColOffsets<RQ, RR>& off,
                                            const uint32_t* rbase, const RowOffsets<RQ, RR>& roff,
                                            uint32_t rdst, bool rpf, int s64, uint4* sB0,
                                            uint4* sB1, int wave, int lane, int col,
                                            uint32_t (&cnt)[RQ][MR]) {
  constexpr int WS = TileCfg<RQ, RR>::WS;
  static_assert(MR == RR || (PB != 0 && TileCfg<RQ, MR>::TC == TileCfg<RQ, RR>::TC &&
                             TileCfg<RQ, MR>::WS == WS),
                "a narrower matching must read the same column stage");
#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int r = 0; r < MR; ++r) cnt[q][r] = 0;

  const int n_stages = (s64 + WS - 1) / WS;
  issue_stage<RQ, RR>(cbase, off, sB0, wave);
  if (rpf) prefetch_round<RQ, RR, 0>(rbase, roff, rdst, wave);
  // One barrier per stage: after it, stage s is in LDS for every wave and
  // every wave has finished matching stage s - 1, whose buffer the copy of
  // stage s + 1 (issued right after the barrier) then overwrites while stage
  // s is matched.  Stages alternate between the two buffers; each pass of
  // this loop runs an even stage from sB0 and the following odd stage from
  // sB1.
  for (int st = 0; st < n_stages; st += 2) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int s = st + half;
      if (s < n_stages) {
        uint4* cur = half ? sB1 : sB0;
        uint4* nxt = half ? sB0 : sB1;
        const int w0 = s * WS;
        wait_vmcnt<0>();
        stage_barrier();
        if (s + 1 < n_stages) {
          issue_stage<RQ, RR>(cbase + (int64_t)(w0 + WS) * (HL * BLK), off, nxt, wave);
          if (rpf) prefetch_round<RQ, RR, 0>(rbase + (int64_t)(w0 + WS) * (HL * BLK), roff, rdst, wave);
        }
        const int nw = (s64 - w0) < WS ? (s64 - w0) : WS;
        if constexpr (PB == 0) {
          match_stage_plain<RQ, MR>(arow, w0, nw, reinterpret_cast<const uint32_t*>(cur), lane,
                                    cnt);
        } else {
          match_stage_pipe<RQ, MR, PB>(arow, w0, nw, cur, col, cnt);
        }
      }
    }
  }
  // every wave is done with both buffers before they are reused
  stage_barrier();
}

// Diagonal tiles of a self pass (upper triangle, i < j): a 64-column block
// of a 64 x 256 tile whose last column precedes the tile's first row holds no
// output pair.  A tile whose first row lies 128 (192) columns past its first
// column matches only its last 2 (1) blocks, with the matching of the
// 32-row (16-row) shape, which reads the same column stage; the skipped
// counts are zero and the epilogue never reads them.  Returns false (and
// does nothing) for any other tile.  Tile-uniform.
template <int RQ, int RR, int PB>
__device__ __forceinline__ bool tile_match_diagonal(CParams* pp, Tile tile, int kk, uint4* sB0,
                                                    uint4* sB1, uint4* sR, int wave, int lane,
                                                    uint32_t (&cnt)[RQ][RR]) {
  static_assert(RQ == 8 && RR == 4 && PB != 0, "64 x 256 pipelined tiles only");
  using Cfg = TileCfg<RQ, RR>;
  if (!pp->self_mode || pp->full_square) return false;
  const int64_t row0 = (int64_t)tile.bi * Cfg::TROWS;
  const int64_t col0 = (int64_t)tile.ct * Cfg::TC;
  const int64_t d = row0 - col0;
  if (d < 2 * 64) return false;
  const int s64 = pp->s64;
  const CU32* arow = (CU32*)(pp->row_stripes +
                             ((int64_t)kk * pp->nb_rows + row0 / BLK) * (int64_t)s64 * (HL * BLK) +
                             row0 % BLK + (wave / Cfg::CG) * RQ);
  const int nb_cols = pp->nb_cols;
  const uint32_t* cbase = pp->col_stripes + (int64_t)kk * nb_cols * (int64_t)s64 * (HL * BLK) +
                          (int64_t)(col0 / BLK) * s64 * (HL * BLK);
  const ColOffsets<RQ, RR> off = col_offsets<RQ, RR>(col0, nb_cols, s64, wave, lane);
  const bool rpf = pp->row_prefetch != 0;
  const uint32_t* rbase = pp->row_stripes +
                          ((int64_t)kk * pp->nb_rows + row0 / BLK) * (int64_t)s64 * (HL * BLK) +
                          row0 % BLK;
  const RowOffsets<RQ, RR> roff = row_offsets<RQ, RR>(wave, lane);
  const uint32_t rdst = lds_addr(sR) + (uint32_t)(wave * 64 * 16);
  if (d >= 3 * 64) {
    uint32_t c1[RQ][1];
    tile_stages<RQ, RR, PB, 1>(arow, cbase, off, rbase, roff, rdst, rpf, s64, sB0, sB1, wave,
                               lane, lane + 3 * 64, c1);
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      cnt[q][0] = cnt[q][1] = cnt[q][2] = 0;
      cnt[q][3] = c1[q][0];
    }
  } else {
    uint32_t c2[RQ][2];
    tile_stages<RQ, RR, PB, 2>(arow, cbase, off, rbase, roff, rdst, rpf, s64, sB0, sB1, wave,
                               lane, lane + 2 * 64, c2);
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      cnt[q][0] = cnt[q][1] = 0;
      cnt[q][2] = c2[q][0];
      cnt[q][3] = c2[q][1];
    }
  }
  return true;
}

// SKIP: diagonal tiles of a self pass go through tile_match_diagonal (only
// the kernels instantiated with it carry that code).
template <int RQ, int RR, int PB, bool SKIP = false>
__device__ __forceinline__ void tile_match(CParams* pp, Tile tile, int kk, uint4* sB0,
                                           uint4* sB1, uint4* sR, int wave, int lane,
                                           uint32_t (&cnt)[RQ][RR]) {
  if constexpr (SKIP) {
    if (tile_match_diagonal<RQ, RR, PB>(pp, tile, kk, sB0, sB1, sR, wave, lane, cnt)) return;
  }
  using Cfg = TileCfg<RQ, RR>;
  constexpr int TC = Cfg::TC;
  constexpr int WS = Cfg::WS;
  constexpr int TROWS = Cfg::TROWS;
  const int s64 = pp->s64;

  // row operands: RQ consecutive samples of this wave, wave-uniform address,
  // read through the constant address space so they are scalar loads into
  // SGPRs (the stripes are never written while a distance kernel runs)
  const int64_t row0 = (int64_t)tile.bi * TROWS;
  const CU32* arow = (CU32*)(pp->row_stripes +
                             ((int64_t)kk * pp->nb_rows + row0 / BLK) * (int64_t)s64 * (HL * BLK) +
                             row0 % BLK + (wave / Cfg::CG) * RQ);
  // the lane's first column within the tile
  const int col_in_tile = (wave % Cfg::CG) * 64 * RR + lane;
  // column slabs of this k-mer length.  The last stage may run past word
  // s64 - 1: the stripe buffer carries zero padding at its end, and those
  // words are never computed on.
  const int64_t col0 = (int64_t)tile.ct * TC;
  const int nb_cols = pp->nb_cols;
  const uint32_t* __restrict__ col_kk =
      pp->col_stripes + (int64_t)kk * nb_cols * (int64_t)s64 * (HL * BLK);

#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int r = 0; r < RR; ++r) cnt[q][r] = 0;

  const int n_stages = (s64 + WS - 1) / WS;
  const ColOffsets<RQ, RR> off = col_offsets<RQ, RR>(col0, nb_cols, s64, wave, lane);
  const uint32_t* cbase = col_kk + (int64_t)(col0 / BLK) * s64 * (HL * BLK);
  const bool rpf = PB != 0 && pp->row_prefetch != 0;
  const uint32_t* rbase = pp->row_stripes +
                          ((int64_t)kk * pp->nb_rows + row0 / BLK) * (int64_t)s64 * (HL * BLK) +
                          row0 % BLK;
  const RowOffsets<RQ, RR> roff = row_offsets<RQ, RR>(wave, lane);
  const uint32_t rdst = lds_addr(sR) + (uint32_t)(wave * 64 * 16);
  issue_stage<RQ, RR>(cbase, off, sB0, wave);
  if (rpf) prefetch_round<RQ, RR, 0>(rbase, roff, rdst, wave);
  // One barrier per stage: after it, stage s is in LDS for every wave and
  // every wave has finished matching stage s - 1, whose buffer the copy of
  // stage s + 1 (issued right after the barrier) then overwrites while stage
  // s is matched.  Stages alternate between the two buffers; each pass of
  // this loop runs an even stage from sB0 and the following odd stage from
  // sB1.
  for (int st = 0; st < n_stages; st += 2) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int s = st + half;
      if (s < n_stages) {
        uint4* cur = half ? sB1 : sB0;
        uint4* nxt = half ? sB0 : sB1;
        const int w0 = s * WS;
        wait_vmcnt<0>();
        stage_barrier();
        if (s + 1 < n_stages) {
          issue_stage<RQ, RR>(cbase + (int64_t)(w0 + WS) * (HL * BLK), off, nxt, wave);
          if (rpf) prefetch_round<RQ, RR, 0>(rbase + (int64_t)(w0 + WS) * (HL * BLK), roff, rdst, wave);
        }
        const int nw = (s64 - w0) < WS ? (s64 - w0) : WS;
        const uint32_t* sB = reinterpret_cast<const uint32_t*>(cur);
        if constexpr (PB == 0) {
          match_stage_plain<RQ, RR>(arow, w0, nw, sB, lane, cnt);
        } else {
          match_stage_pipe<RQ, RR, PB>(arow, w0, nw, cur, col_in_tile, cnt);
        }
      }
    }
  }
  // every wave is done with both buffers before they are reused
  stage_barrier();
}

// Counts of this wave / lane into a tile count block [n_k][rows][cols].
template <int RQ, int RR>
__device__ __forceinline__ void store_counts(uint16_t* tile_counts, int kk, int wave, int lane,
                                             const uint32_t (&cnt)[RQ][RR]) {
  using Cfg = TileCfg<RQ, RR>;
  constexpr int TC = Cfg::TC;
  uint16_t* cbase = tile_counts + ((int64_t)kk * Cfg::TROWS + (wave / Cfg::CG) * RQ) * TC +
                    (wave % Cfg::CG) * 64 * RR + lane;
#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int r = 0; r < RR; ++r) cbase[q * TC + 64 * r] = (uint16_t)cnt[q][r];
}

// ---------------------------------------------------------------------------
// The tile kernel: one (tile, k-mer length) item per workgroup.
// ---------------------------------------------------------------------------
template <int RQ, int RR, int PB>
__global__ __launch_bounds__(WAVES * 64, 4) void dist_tiles(DistParams p) {
  using Cfg = TileCfg<RQ, RR>;
  __shared__ uint4 sB0[Cfg::STAGE_U4];
  __shared__ uint4 sB1[Cfg::STAGE_U4];
  __shared__ uint4 sR[PB ? Cfg::ROW_LDS_U4 : 64];  // row prefetch: pipelined shapes only
  __shared__ int s_last;
  __shared__ int s_stop;
  // the parameters are the kernel's only argument: scalar loads straight
  // from the kernarg segment (no copy)
  CParams* pp = (CParams*)__builtin_amdgcn_kernarg_segment_ptr();

  const int64_t item = p.item_base + blockIdx.x;
  const int64_t t = item / p.n_k;
  const int kk = (int)(item - t * p.n_k);
  Tile tile = p.tiles[t];
  // wave-uniform values (kept in SGPRs)
  tile.bi = __builtin_amdgcn_readfirstlane(tile.bi);
  tile.ct = __builtin_amdgcn_readfirstlane(tile.ct);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  // a cancelled call skips the matching; one read per workgroup, shared, so
  // that every wave takes the same branch (the matching has barriers)
  if (threadIdx.x == 0) s_stop = cancel_seen(p.ctl.cancel) ? 1 : 0;
  __syncthreads();
  const int stop = __builtin_amdgcn_readfirstlane(s_stop);

  // per-tile count scratch: [tile][kk][row][col]
  uint16_t* tile_counts = p.counts + t * p.n_k * (int64_t)(Cfg::TROWS * Cfg::TC);
  if (!stop) {
    uint32_t cnt[RQ][RR];
    tile_match<RQ, RR, PB>(pp, tile, kk, sB0, sB1, sR, wave, lane, cnt);
    store_counts<RQ, RR>(tile_counts, kk, wave, lane, cnt);
  }

  // completion: the last workgroup of this tile runs the epilogue (unless
  // the call was cancelled, which then holds for every later read)
  __threadfence();
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned prev = atomicAdd(&p.tile_done[t], 1u);
    const bool last = prev == (unsigned)(p.n_k - 1);
    s_last = last ? (cancel_seen(p.ctl.cancel) ? 2 : 1) : 0;
    if (last) p.tile_done[t] = 0;  // ready for the next launch
  }
  __syncthreads();
  if (s_last != 1) return;
  __threadfence();
  tile_epilogue<RQ, RR>(pp, tile_counts, tile, wave, lane);
  if (threadIdx.x == 0) add_progress(p.ctl, (unsigned long long)p.n_k);
}

// dist_tiles<8, 4, 2> for the (tile, k) items of a self pass's diagonal tiles:
// the column blocks that hold no output pair are skipped (tile_match_diagonal);
// any other tile runs as in dist_tiles.  A kernel of its own, so that the code
// of dist_tiles itself does not change with it.
__global__ __launch_bounds__(WAVES * 64, 4) void dist_tiles_diagonal(DistParams p) {
  constexpr int RQ = 8, RR = 4, PB = 2;
  using Cfg = TileCfg<RQ, RR>;
  __shared__ uint4 sB0[Cfg::STAGE_U4];
  __shared__ uint4 sB1[Cfg::STAGE_U4];
  __shared__ uint4 sR[PB ? Cfg::ROW_LDS_U4 : 64];  // row prefetch: pipelined shapes only
  __shared__ int s_last;
  __shared__ int s_stop;
  // the parameters are the kernel's only argument: scalar loads straight
  // from the kernarg segment (no copy)
  CParams* pp = (CParams*)__builtin_amdgcn_kernarg_segment_ptr();

  const int64_t item = p.item_base + blockIdx.x;
  const int64_t t = item / p.n_k;
  const int kk = (int)(item - t * p.n_k);
  Tile tile = p.tiles[t];
  // wave-uniform values (kept in SGPRs)
  tile.bi = __builtin_amdgcn_readfirstlane(tile.bi);
  tile.ct = __builtin_amdgcn_readfirstlane(tile.ct);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  // a cancelled call skips the matching; one read per workgroup, shared, so
  // that every wave takes the same branch (the matching has barriers)
  if (threadIdx.x == 0) s_stop = cancel_seen(p.ctl.cancel) ? 1 : 0;
  __syncthreads();
  const int stop = __builtin_amdgcn_readfirstlane(s_stop);

  // per-tile count scratch: [tile][kk][row][col]
  uint16_t* tile_counts = p.counts + t * p.n_k * (int64_t)(Cfg::TROWS * Cfg::TC);
  if (!stop) {
    uint32_t cnt[RQ][RR];
    tile_match<RQ, RR, PB, true>(pp, tile, kk, sB0, sB1, sR, wave, lane, cnt);
    store_counts<RQ, RR>(tile_counts, kk, wave, lane, cnt);
  }

  // completion: the last workgroup of this tile runs the epilogue (unless
  // the call was cancelled, which then holds for every later read)
  __threadfence();
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned prev = atomicAdd(&p.tile_done[t], 1u);
    const bool last = prev == (unsigned)(p.n_k - 1);
    s_last = last ? (cancel_seen(p.ctl.cancel) ? 2 : 1) : 0;
    if (last) p.tile_done[t] = 0;  // ready for the next launch
  }
  __syncthreads();
  if (s_last != 1) return;
  __threadfence();
  tile_epilogue<RQ, RR>(pp, tile_counts, tile, wave, lane);
  if (threadIdx.x == 0) add_progress(p.ctl, (unsigned long long)p.n_k);
}

// ---------------------------------------------------------------------------
// Persistent batch kernel: many query-vs-ref jobs (each with its own sets,
// k-mer lengths, sketch size and output) in one launch.  Work items are
// whole tiles (every k-mer length of the tile, then its epilogue) taken from
// NQ queues; workgroup b starts on queue b % NQ (the XCD it is dispatched
// to) and, once that queue is drained, moves on to the next ones in turn,
// never returning to a drained queue; it exits after the last one.  Counts
// go to the workgroup's own scratch block and are read back by the same
// lanes in the epilogue, so no cross-workgroup synchronisation is needed.
// ---------------------------------------------------------------------------
// LDS of the persistent kernels' matching: one set, sized for the largest
// tile shape (64 x 256) and shared by every shape a kernel runs, so a kernel
// that mixes shapes holds it once.  Every batch shape stages the same
// 28 KiB column stage (4 / RR words of 64 RR columns); the row prefetch
// area grows with the tile rows.
__shared__ uint4 g_batch_sB0[TileCfg<8, 4>::STAGE_U4];
__shared__ uint4 g_batch_sB1[TileCfg<8, 4>::STAGE_U4];
__shared__ uint4 g_batch_sR[TileCfg<8, 4>::ROW_LDS_U4];

// One (tile, k-mer length) of a batch item: counts into the workgroup's
// scratch block.  Out of line so that the matching loop is register-allocated
// on its own, exactly as in dist_tiles, instead of around the persistent
// loop's state (which would push the counts out to scratch memory on every
// word).  Arguments arrive in VGPRs and are made wave-uniform again here.
template <int RQ, int RR, int PB>
__device__ __noinline__ void batch_tile_k(CParams* pp_in, int bi_in, int ct_in, int kk_in,
                                          uint16_t* scratch_in) {
  using Cfg = TileCfg<RQ, RR>;
  static_assert(Cfg::STAGE_U4 == TileCfg<8, 4>::STAGE_U4 &&
                    Cfg::ROW_LDS_U4 <= TileCfg<8, 4>::ROW_LDS_U4,
                "batch shapes share the LDS stage buffers");
  uint4* sB0 = g_batch_sB0;
  uint4* sB1 = g_batch_sB1;
  uint4* sR = g_batch_sR;
  const uint64_t pv = (uint64_t)(uintptr_t)pp_in;
  const uint32_t plo = __builtin_amdgcn_readfirstlane((uint32_t)pv);
  const uint32_t phi = __builtin_amdgcn_readfirstlane((uint32_t)(pv >> 32));
  CParams* pp = (CParams*)(uintptr_t)(((uint64_t)phi << 32) | plo);
  const uint64_t sv = (uint64_t)(uintptr_t)scratch_in;
  const uint32_t slo = __builtin_amdgcn_readfirstlane((uint32_t)sv);
  const uint32_t shi = __builtin_amdgcn_readfirstlane((uint32_t)(sv >> 32));
  uint16_t* scratch = (uint16_t*)(uintptr_t)(((uint64_t)shi << 32) | slo);
  Tile tile;
  tile.bi = __builtin_amdgcn_readfirstlane(bi_in);
  tile.ct = __builtin_amdgcn_readfirstlane(ct_in);
  const int kk = __builtin_amdgcn_readfirstlane(kk_in);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  uint32_t cnt[RQ][RR];
  tile_match<RQ, RR, PB>(pp, tile, kk, sB0, sB1, sR, wave, lane, cnt);
  store_counts<RQ, RR>(scratch, kk, wave, lane, cnt);
}

template <int RQ, int RR, int PB>
__global__ __launch_bounds__(WAVES * 64, 4) void dist_batch(BatchArgs a) {
  using Cfg = TileCfg<RQ, RR>;
  __shared__ int64_t s_item;
  __shared__ int s_tried;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int home = (int)(blockIdx.x % BATCH_QUEUES);
  uint16_t* scratch =
      a.scratch + (int64_t)blockIdx.x * a.max_k * (int64_t)(Cfg::TROWS * Cfg::TC);
  int tried = 0;  // queues found drained so far (workgroup-uniform)
  for (;;) {
    if (threadIdx.x == 0) {
      int64_t got = -1;
      if (cancel_seen(a.ctl.cancel)) tried = BATCH_QUEUES;  // cancelled: take no more items
      while (tried < BATCH_QUEUES) {
        const int q = (home + tried) % BATCH_QUEUES;
        const int64_t size = a.queue_begin[q + 1] - a.queue_begin[q];
        const unsigned idx = atomicAdd(&a.queue_next[q], 1u);
        if ((int64_t)idx < size) {
          got = a.queue_begin[q] + idx;
          break;
        }
        ++tried;
      }
      s_item = got;
      s_tried = tried;
    }
    __syncthreads();
    const int64_t it = s_item;
    tried = s_tried;
    __syncthreads();  // s_item is rewritten only after every thread read it
    if (it < 0) break;
    const BatchItem bi = a.items[it];
    const int job = __builtin_amdgcn_readfirstlane(bi.job);
    Tile tile;
    tile.bi = __builtin_amdgcn_readfirstlane(bi.bi);
    tile.ct = __builtin_amdgcn_readfirstlane(bi.ct);
    CParams* pp = (CParams*)(a.jobs + job);
    const int n_k = pp->n_k;
    for (int kk = 0; kk < n_k; ++kk) batch_tile_k<RQ, RR, PB>(pp, tile.bi, tile.ct, kk, scratch);
    tile_epilogue<RQ, RR>(pp, scratch, tile, wave, lane);
    if (threadIdx.x == 0) add_progress(a.ctl, (unsigned long long)n_k);
  }
}

// One whole tile of a batch item in shape RQ x RR: every k-mer length into
// the workgroup's scratch block, then the epilogue, then progress.  Out of
// line: the mixed-shape kernel's frame then only dispatches (a few of its
// values are saved around the calls).
template <int RQ, int RR, int PB>
__device__ __noinline__ void batch_tile(CParams* pp, Tile tile, uint16_t* scratch, Control ctl,
                                        int wave, int lane) {
  const int n_k = pp->n_k;
  for (int kk = 0; kk < n_k; ++kk) batch_tile_k<RQ, RR, PB>(pp, tile.bi, tile.ct, kk, scratch);
  tile_epilogue<RQ, RR>(pp, scratch, tile, wave, lane);
  if (threadIdx.x == 0) add_progress(ctl, (unsigned long long)n_k);
}

// The persistent kernel of dist_batch with a tile shape per item (item.pad:
// 2 = 64 x 256, 4 = 32 x 256, 5 = 16 x 256), so that each job of a batch can
// cover its rows with the tile heights that waste the least of its work on
// padding rows.  The shapes share the LDS stage buffers; a workgroup's
// scratch block holds the counts of the largest shape.
__global__ __launch_bounds__(WAVES * 64, 4) void dist_batch_mixed(BatchArgs a) {
  __shared__ int64_t s_item;
  __shared__ int s_tried;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int home = (int)(blockIdx.x % BATCH_QUEUES);
  uint16_t* scratch = a.scratch + (int64_t)blockIdx.x * a.max_k *
                                      (int64_t)(TileCfg<8, 4>::TROWS * TileCfg<8, 4>::TC);
  int tried = 0;  // queues found drained so far (workgroup-uniform)
  for (;;) {
    if (threadIdx.x == 0) {
      int64_t got = -1;
      if (cancel_seen(a.ctl.cancel)) tried = BATCH_QUEUES;  // cancelled: take no more items
      while (tried < BATCH_QUEUES) {
        const int q = (home + tried) % BATCH_QUEUES;
        const int64_t size = a.queue_begin[q + 1] - a.queue_begin[q];
        const unsigned idx = atomicAdd(&a.queue_next[q], 1u);
        if ((int64_t)idx < size) {
          got = a.queue_begin[q] + idx;
          break;
        }
        ++tried;
      }
      s_item = got;
      s_tried = tried;
    }
    __syncthreads();
    const int64_t it = s_item;
    tried = s_tried;
    __syncthreads();  // s_item is rewritten only after every thread read it
    if (it < 0) break;
    const BatchItem bi = a.items[it];
    const int job = __builtin_amdgcn_readfirstlane(bi.job);
    const int shape = __builtin_amdgcn_readfirstlane(bi.pad);
    Tile tile;
    tile.bi = __builtin_amdgcn_readfirstlane(bi.bi);
    tile.ct = __builtin_amdgcn_readfirstlane(bi.ct);
    CParams* pp = (CParams*)(a.jobs + job);
    if (shape == 5) {
      batch_tile<8, 1, 2>(pp, tile, scratch, a.ctl, wave, lane);
    } else if (shape == 4) {
      batch_tile<8, 2, 2>(pp, tile, scratch, a.ctl, wave, lane);
    } else {
      batch_tile<8, 4, 2>(pp, tile, scratch, a.ctl, wave, lane);
    }
  }
}

// ---------------------------------------------------------------------------
// Split passes: dist_items counts matches, dist_items_out turns the counts
// into output.
//
// A workgroup of dist_items takes one item: a tile, one k-mer length and all or
// one run of that sketch's words, and stores its match counts as a block of
// its own.  (Tile, k-mer length) pairs that fill whole rounds of the 512
// resident workgroups are one item each; the others, all of them in a small
// pass, are cut into the runs of words that make their rounds shortest
// (cut_items in the host layer), so that a pass of few tiles spreads over
// every CU and a large one has no idle last round.  One item over 156 words
// takes 0.68 ms by itself, however small the pass: calls on 48 genomes went
// from 774 to 148 us, one query against 6,000 references from 756 to 255 us
// (8 k-mer lengths, 10,000 bins).
//
// Tiles are 64, 32 or 16 rows high, so that the rows past the last multiple
// of 64 are covered without computing whole tiles of padding.
//
// Workgroup b of a part of n items takes item (b % 8) * ceil(n / 8) + b / 8:
// consecutive workgroups go to the 8 XCDs in turn, so each XCD walks one
// contiguous eighth of the list and keeps the row and column panels its tiles
// share in its own L2.
// ---------------------------------------------------------------------------
struct ItemAt {
  int tile, kk;
  int unit0, units;  // words or halves
  int64_t block;     // of the counts
};

// The item of this workgroup; false: none (padding of the last eighth).
__device__ __forceinline__ bool item_at(const ItemArgs& a, int n_k, int units, ItemAt& it) {
  int b = (int)blockIdx.x, n = a.whole;
  const int first = (n + BATCH_QUEUES - 1) / BATCH_QUEUES * BATCH_QUEUES;
  const bool whole = b < first;
  if (!whole) {
    b -= first;
    n = a.n_items - a.whole;
  }
  const int per = (n + BATCH_QUEUES - 1) / BATCH_QUEUES;
  const int x = b % BATCH_QUEUES * per + b / BATCH_QUEUES;
  if (b / BATCH_QUEUES >= per || x >= n) return false;
  int pair = x;
  it.unit0 = 0;
  it.units = units;
  it.block = x;
  if (!whole) {
    const int pairs = n / a.runs;
    const int run = x / pairs;
    pair = a.whole + (x - run * pairs);
    it.unit0 = run * a.run_units;
    it.units = min(a.run_units, units - it.unit0);
    it.block = a.whole + (int64_t)(x - run * pairs) * a.runs + run;
  }
  const int tall = a.n_tall * n_k;
  const int at = pair < tall ? pair : pair - tall;
  const int per_k = pair < tall ? a.n_tall : a.n_tiles - a.n_tall;
  it.kk = at / per_k;
  it.tile = at - it.kk * per_k + (pair < tall ? 0 : a.n_tall);
  return true;
}

// Number of the pair (tile t, k-mer length k).
__device__ __forceinline__ int item_pair(const ItemArgs& a, int n_k, int t, int k) {
  return t < a.n_tall ? k * a.n_tall + t
                      : a.n_tall * n_k + k * (a.n_tiles - a.n_tall) + t - a.n_tall;
}

template <int RR>
__device__ __forceinline__ void match_item(CParams* pp, int row0, int ct, int kk, int w0, int nw,
                                           uint4* sB0, uint4* sB1, uint4* sR, uint16_t* counts,
                                           int wave, int lane) {
  constexpr int RQ = 8, PB = 2;
  using Cfg = TileCfg<RQ, RR>;
  const int s64 = pp->s64;
  const int nb_cols = pp->nb_cols;
  const int64_t word0 = (int64_t)w0 * (HL * BLK);
  const uint32_t* rbase =
      pp->row_stripes + ((int64_t)kk * pp->nb_rows + row0 / BLK) * (int64_t)s64 * (HL * BLK) +
      word0 + row0 % BLK;
  const CU32* arow = (CU32*)(rbase + (wave / Cfg::CG) * RQ);
  const int64_t col0 = (int64_t)ct * Cfg::TC;
  const uint32_t* cbase =
      pp->col_stripes + ((int64_t)kk * nb_cols + col0 / BLK) * (int64_t)s64 * (HL * BLK) + word0;
  const ColOffsets<RQ, RR> off = col_offsets<RQ, RR>(col0, nb_cols, s64, wave, lane);
  const RowOffsets<RQ, RR> roff = row_offsets<RQ, RR>(wave, lane);
  const uint32_t rdst = lds_addr(sR) + (uint32_t)(wave * 64 * 16);
  uint32_t cnt[RQ][RR];
  tile_stages<RQ, RR, PB, RR>(arow, cbase, off, rbase, roff, rdst, pp->row_prefetch != 0, nw, sB0,
                              sB1, wave, lane, (wave % Cfg::CG) * 64 * RR + lane, cnt);
  store_counts<RQ, RR>(counts, 0, wave, lane, cnt);
}

__global__ __launch_bounds__(WAVES * 64, 4) void dist_items(DistParams p, ItemArgs a) {
  __shared__ uint4 sB0[TileCfg<8, 4>::STAGE_U4];
  __shared__ uint4 sB1[TileCfg<8, 4>::STAGE_U4];
  __shared__ uint4 sR[TileCfg<8, 4>::ROW_LDS_U4];
  __shared__ int s_stop;
  // both arguments are read with scalar loads from the kernarg segment
  CParams* pp = (CParams*)__builtin_amdgcn_kernarg_segment_ptr();
  ItemAt it;
  if (!item_at(a, p.n_k, p.s64, it)) return;
  if (p.ctl.stop != nullptr && blockIdx.x >= (uint32_t)a.unwatched) {
    // a cancelled call skips the matching; one read per workgroup, shared, so
    // that every wave takes the same branch (the matching has barriers)
    if (threadIdx.x == 0) s_stop = item_stopped(p.ctl, blockIdx.x) ? 1 : 0;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_stop)) return;
  }
  const ItemTile tile = a.tiles[it.tile];
  const int row0 = __builtin_amdgcn_readfirstlane(tile.row0);
  const int ct = __builtin_amdgcn_readfirstlane(tile.ct);
  const int rows = __builtin_amdgcn_readfirstlane(tile.rows);
  const int kk = it.kk, w0 = it.unit0, nw = it.units;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  uint16_t* counts = p.counts + it.block * ITEM_COUNTS;
  if (rows == 64) {
    match_item<4>(pp, row0, ct, kk, w0, nw, sB0, sB1, sR, counts, wave, lane);
  } else if (rows == 32) {
    match_item<2>(pp, row0, ct, kk, w0, nw, sB0, sB1, sR, counts, wave, lane);
  } else {
    match_item<1>(pp, row0, ct, kk, w0, nw, sB0, sB1, sR, counts, wave, lane);
  }
  if (threadIdx.x == 0) add_item(p.ctl);
}

// Counts of OUT_K k-mer lengths from their runs' blocks, x[i] at the pair's
// count in the first block: 4 runs of all lengths at a time.
__device__ __forceinline__ void sum_runs(const uint16_t* const (&x)[OUT_K],
                                         const int (&runs)[OUT_K], uint32_t (&c)[OUT_K]) {
  int most = 1;
#pragma unroll
  for (int i = 0; i < OUT_K; ++i) {
    most = max(most, runs[i]);
    c[i] = 0;
  }
  for (int y = 0; y < most; y += 4) {
    uint32_t v[4][OUT_K];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < OUT_K; ++i) {
        v[j][i] = y + j < runs[i] ? x[i][(int64_t)(y + j) * ITEM_COUNTS] : 0u;
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < OUT_K; ++i) c[i] += v[j][i];
  }
}

// Output of a split pass: one lane per pair, a.out_rows rows of one tile per
// workgroup (1 in a small pass, so that no lane has to do four), the 256
// columns of a row read and written side by side.  Left to the last workgroup
// of each tile, as dist_tiles does it, the epilogue of a tile runs 32 pairs per
// lane one after the other on one CU: the 2.1M pairs of 2,050 samples x 13
// k-mer lengths of 1,024 bins (Jaccards) took 3.58 ms that way and take 0.67 ms
// here (whole calls).
__global__ __launch_bounds__(256) void dist_items_out(DistParams p, ItemArgs a) {
  CParams* pp = (CParams*)__builtin_amdgcn_kernarg_segment_ptr();
  CParams& q = *pp;
  const int parts = 64 / a.out_rows;
  const int t = (int)(blockIdx.x / parts);
  const int r0 = (int)(blockIdx.x % parts) * a.out_rows;
  const ItemTile tile = a.tiles[t];
  if (r0 >= tile.rows) return;
  const int64_t gj = (int64_t)tile.ct * 256 + threadIdx.x;
  const double bins = 64.0 * (double)q.s64;
  const double rbins = 1.0 / bins;
  for (int r = r0; r < r0 + a.out_rows; ++r) {
    const int64_t gi = tile.row0 + r;
    if (!pair_valid(q, gi, gj)) continue;
    const uint16_t* cp = q.counts + r * 256 + threadIdx.x;
    pair_output(q, gi, gj, bins, rbins, [&](int k0, uint32_t (&c)[OUT_K]) {
      const uint16_t* x[OUT_K];
      int runs[OUT_K];
#pragma unroll
      for (int i = 0; i < OUT_K; ++i) {
        const int pair = item_pair(a, q.n_k, t, min(k0 + i, q.n_k - 1));
        const bool whole = pair < a.whole;
        x[i] = cp + (whole ? pair : a.whole + (int64_t)(pair - a.whole) * a.runs) * ITEM_COUNTS;
        runs[i] = whole ? 1 : a.runs;
      }
      sum_runs(x, runs, c);
    });
  }
}

static unsigned item_grid(const ItemArgs& a) {
  const int per1 = (a.whole + BATCH_QUEUES - 1) / BATCH_QUEUES;
  const int per2 = (a.n_items - a.whole + BATCH_QUEUES - 1) / BATCH_QUEUES;
  return (unsigned)((per1 + per2) * BATCH_QUEUES);
}

// The items of a batch: the same matching over the tiles of many jobs, each
// job's parameters from the batch's table.  12 jobs of 1 to 512 queries x
// 375 to 3,000 references as whole tiles of the persistent kernel (every
// k-mer length of a tile on one workgroup) took 2.83 ms, its last tiles alone
// on their CUs; as items and the output kernel (0.17 ms) 1.88 ms.
__global__ __launch_bounds__(WAVES * 64, 4) void dist_batch_items(BatchItemArgs a) {
  __shared__ uint4 sB0[TileCfg<8, 4>::STAGE_U4];
  __shared__ uint4 sB1[TileCfg<8, 4>::STAGE_U4];
  __shared__ uint4 sR[TileCfg<8, 4>::ROW_LDS_U4];
  __shared__ int s_stop;
  const BatchRun it = a.items[blockIdx.x];
  const int t = __builtin_amdgcn_readfirstlane(it.tile);
  if (t < 0) return;
  if (a.ctl.stop != nullptr && blockIdx.x >= ITEM_SLOTS) {
    if (threadIdx.x == 0) s_stop = item_stopped(a.ctl, blockIdx.x) ? 1 : 0;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_stop)) return;
  }
  const BatchTile tile = a.tiles[t];
  const int job = __builtin_amdgcn_readfirstlane(tile.job);
  const int row0 = __builtin_amdgcn_readfirstlane(tile.row0);
  const int ct = __builtin_amdgcn_readfirstlane(tile.ct);
  const int rows = __builtin_amdgcn_readfirstlane(tile.rows);
  const int kk = __builtin_amdgcn_readfirstlane(it.kk);
  const int w0 = __builtin_amdgcn_readfirstlane(it.word0);
  const int nw = __builtin_amdgcn_readfirstlane(it.words);
  const int block = __builtin_amdgcn_readfirstlane(it.block);
  CParams* pp = (CParams*)(a.jobs + job);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  uint16_t* counts = a.counts + (int64_t)block * ITEM_COUNTS;
  if (rows == 64) {
    match_item<4>(pp, row0, ct, kk, w0, nw, sB0, sB1, sR, counts, wave, lane);
  } else if (rows == 32) {
    match_item<2>(pp, row0, ct, kk, w0, nw, sB0, sB1, sR, counts, wave, lane);
  } else {
    match_item<1>(pp, row0, ct, kk, w0, nw, sB0, sB1, sR, counts, wave, lane);
  }
  if (threadIdx.x == 0) add_item(a.ctl);
}

__global__ __launch_bounds__(256) void dist_batch_items_out(BatchItemArgs a) {
  const int parts = 64 / a.out_rows;
  const BatchTile tile = a.tiles[blockIdx.x / parts];
  const int r0 = (int)(blockIdx.x % parts) * a.out_rows;
  if (r0 >= tile.rows) return;
  CParams& q = *(CParams*)(a.jobs + __builtin_amdgcn_readfirstlane(tile.job));
  const int64_t gj = (int64_t)tile.ct * 256 + threadIdx.x;
  const double bins = 64.0 * (double)q.s64;
  const double rbins = 1.0 / bins;
  for (int r = r0; r < r0 + a.out_rows; ++r) {
    const int64_t gi = tile.row0 + r;
    if (!pair_valid(q, gi, gj)) continue;
    const uint16_t* cp = a.counts + (int64_t)tile.block0 * ITEM_COUNTS + r * 256 + threadIdx.x;
    pair_output(q, gi, gj, bins, rbins, [&](int k0, uint32_t (&c)[OUT_K]) {
      const uint16_t* x[OUT_K];
      int runs[OUT_K];
#pragma unroll
      for (int i = 0; i < OUT_K; ++i) {
        x[i] = cp + (int64_t)min(k0 + i, q.n_k - 1) * tile.runs * ITEM_COUNTS;
        runs[i] = tile.runs;
      }
      sum_runs(x, runs, c);
    });
  }
}

hipError_t launch_batch_items(const BatchItemArgs& a, hipStream_t stream) {
  if (a.n_items <= 0) return hipSuccess;
  dist_batch_items<<<(unsigned)a.n_items, WAVES * 64, 0, stream>>>(a);
  dist_batch_items_out<<<(unsigned)(a.n_tiles * (64 / a.out_rows)), 256, 0, stream>>>(a);
  return hipGetLastError();
}

hipError_t launch_items(const DistParams& p, const ItemArgs& a, hipStream_t stream) {
  if (a.n_items <= 0) return hipSuccess;
  dist_items<<<item_grid(a), WAVES * 64, 0, stream>>>(p, a);
  dist_items_out<<<(unsigned)(a.n_tiles * (64 / a.out_rows)), 256, 0, stream>>>(p, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Coded passes: fewer bit planes per pair.
//
// A group of at most CODE_ROWS rows holds V distinct values at a bin, V far
// below the 2^14 a 14-bit value could take (at most CODE_ROWS; 110-170 in 8,192
// tree samples, about 750 in unrelated ones, whose 10 planes still beat 14: 30.0
// ms against 33.8), so equality with a row is decided by the value's rank among those
// V: code 1 .. V for a value some row of the group holds, 0 for any other.
// Two codes are equal exactly when the values are, as one of them is always a
// row's; the match counts are the same whole numbers.  A run of 32 bins
// ("half", one dword of the sketch words) then needs only the planes of its
// largest code (its width, 3 .. CODE_PLANES) instead of 14: width + 1 VALU
// operations per pair and half instead of 15.
//
// code_kernel, one workgroup per (group, k-mer length, half), builds the
// ranks in LDS: per bin a bitmap of the 2^14 values (512 dwords, a row's value
// sets one bit) and beside each dword the number of values set in the dwords
// before it (8 bytes an entry, 4 KiB a bin, 128 KiB for the half).  A code is
// one 8-byte read, a shift, a population count and an add.  Samples arrive and
// leave bit-sliced; a 16 x 16 bit transpose of both dword halves at once turns
// the 14 planes of a lane's sample into its 32 values and the 32 codes into
// planes.  Bound by VALU: 465 instructions per sample and half (of 32 bins),
// 69% of the time issuing, with about 3 bytes per sample and bin beside it;
// shared by the group's rows that is under one operation per pair and half,
// against the 6 or 7 it saves.  8,192 samples against themselves: coding 3.1 ms
// and matching 21.8 ms (90% of the VALU issue rate, 9 operations per pair and
// half) instead of 34.4 ms; the call 34.9 -> 26.3 ms, kNN of 3,000 5.5 -> 4.6
// ms, 451 queries x 6,000 3.26 -> 2.45 ms.
//
// Codes: [k-mer length][block of 256 samples][half][CODE_PLANES][256] dwords
// per group, each half using its first `width` planes.
// ---------------------------------------------------------------------------
constexpr int CODE_TB = 1024;
constexpr int CODE_SLOT = CODE_PLANES * 256;  // dwords of one (block, half)

__device__ __forceinline__ uint32_t bit_select(uint32_t m, uint32_t a, uint32_t b) {
  return (a & m) | (b & ~m);
}

// One stage of the transpose below: swaps bit blocks of side S.
template <int N, int S>
__device__ __forceinline__ void transpose_stage(uint32_t (&x)[16]) {
  constexpr uint32_t m = S == 4 ? 0x0F0F0F0Fu : (S == 2 ? 0x33333333u : 0x55555555u);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if ((i & S) == 0) {
      const uint32_t a = x[i], b = x[i + S];
      x[i] = bit_select(m, a, b << S);
      x[i + S] = bit_select(m, a >> S, b);
    }
  }
}

// Transposes the two 16 x 16 bit matrices held in the low and the high 16
// bits of x[0..15] (bit j of x[i] <-> bit i of x[j]); its own inverse.  N: only
// x[0..N-1] is needed of the result (N = 8 or 16).
template <int N>
__device__ __forceinline__ void transpose16(uint32_t (&x)[16]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t a = x[i], b = x[i + 8];
    x[i] = __builtin_amdgcn_perm(b, a, 0x06020400u);
    if (N > 8) x[i + 8] = __builtin_amdgcn_perm(b, a, 0x07030501u);
  }
  transpose_stage<N, 4>(x);
  transpose_stage<N, 2>(x);
  transpose_stage<N, 1>(x);
}

// (device-memory pointers of the kernel's tables: without the address space
// the compiler writes through flat stores, which also wait for LDS)
typedef __attribute__((address_space(1))) uint32_t GU32;

// The 14 planes of a sample at one half; transposed, its 32 values: bins i
// (low 16 bits of x[i]) and 16 + i (high 16 bits).
__device__ __forceinline__ void load_planes(const GU32* planes, uint32_t (&x)[BBITS]) {
#pragma unroll
  for (int l = 0; l < BBITS; ++l) x[l] = planes[l * BLK];
}

__device__ __forceinline__ void to_values(const uint32_t (&pl)[BBITS], uint32_t (&x)[16]) {
#pragma unroll
  for (int l = 0; l < BBITS; ++l) x[l] = pl[l];
  x[14] = x[15] = 0;
  transpose16<16>(x);
}

struct CodeSet {  // samples to code: [s0, s1) of a set
  const GU32* planes;    // (kk, block 0, word, plane 0 of the half)
  int64_t block_stride;  // dwords between 128-sample blocks
  GU32* out;             // (kk, block b0, half)
  int64_t out_stride;    // dwords between 256-sample blocks
  int b0;
  int s0, s1;
};

__device__ __forceinline__ const GU32* code_source(const CodeSet& cs, int s) {
  return cs.planes + (int64_t)(s / BLK) * cs.block_stride + s % BLK;
}

// pl: the planes of the lane's first sample, already loaded; the next sample's
// are loaded while one is looked up.
template <int N>
__device__ __forceinline__ void code_samples(const CodeSet& cs, const uint2* tab, int width,
                                             uint32_t (&pl)[BBITS]) {
  for (int s = cs.s0 + (int)threadIdx.x; s < cs.s1; s += CODE_TB) {
    uint32_t x[16];
    to_values(pl, x);
    load_planes(code_source(cs, min(s + CODE_TB, cs.s1 - 1)), pl);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t v0 = x[i] & 0xFFFFu, v1 = x[i] >> 16;
      const uint2 e0 = tab[i * 512 + (v0 >> 5)];
      const uint2 e1 = tab[(16 + i) * 512 + (v1 >> 5)];
      // the bit of value v is bit 31 - v % 32 of its dword: shifted up to
      // bit 31, the sign says whether it is set and the population count is
      // its rank in the dword
      const uint32_t t0 = e0.x << (v0 & 31), t1 = e1.x << (v1 & 31);
      const uint32_t c0 = (uint32_t)((int32_t)t0 >> 31) & (e0.y + __popc(t0));
      const uint32_t c1 = (uint32_t)((int32_t)t1 >> 31) & (e1.y + __popc(t1));
      x[i] = c0 | (c1 << 16);
    }
    transpose16<N>(x);
    GU32* o = cs.out + (s / 256 - cs.b0) * cs.out_stride + s % 256;
#pragma unroll
    for (int l = 0; l < (N < CODE_PLANES ? N : CODE_PLANES); ++l) {
      if (l < width) o[l * 256] = x[l];
    }
  }
}

// Sum of x over the lanes up to and including this one.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t x) {
  // row_shr 1, 2, 4, 8 inside the rows of 16 lanes, then the row totals
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);  // row_bcast15
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);  // row_bcast31
  return x;
}

// One (group, k-mer length, half) of a coding launch.
struct CodeItem {
  int kh;
  CodeSet rows, cols;
  GU32* widths;
  bool apart;  // rows coded apart from the columns
};

__device__ __forceinline__ CodeItem code_item(const DistParams& p, const CodeGroup* groups,
                                              int n_groups, int item) {
  const CodeGroup cg = groups[item % n_groups];
  CodeItem it;
  it.kh = item / n_groups;
  const int halves = 2 * p.s64;
  const int kk = it.kh / halves;
  const int half = it.kh - kk * halves;
  const int64_t rblock = (int64_t)p.s64 * (HL * BLK);
  const int64_t at = (int64_t)(half >> 1) * (HL * BLK) + (half & 1) * (BBITS * BLK);
  const int64_t out_stride = (int64_t)halves * CODE_SLOT;
  it.cols.planes = (const GU32*)p.col_stripes + (int64_t)kk * p.nb_cols * rblock + at;
  it.cols.block_stride = rblock;
  it.cols.out = (GU32*)cg.cols + (int64_t)kk * cg.ncb * out_stride + (int64_t)half * CODE_SLOT;
  it.cols.out_stride = out_stride;
  it.cols.b0 = cg.cb0;
  it.cols.s0 = cg.cb0 * 256;
  it.cols.s1 = min(p.nb_cols * BLK, (cg.cb0 + cg.ncb) * 256);
  it.rows = it.cols;
  it.rows.planes = (const GU32*)p.row_stripes + (int64_t)kk * p.nb_rows * rblock + at;
  it.rows.out = (GU32*)cg.rows + (int64_t)kk * cg.nrb * out_stride + (int64_t)half * CODE_SLOT;
  it.rows.b0 = cg.rb0;
  it.rows.s0 = cg.row0;
  it.rows.s1 = cg.row0 + cg.n_rows;
  it.widths = (GU32*)cg.widths;
  it.apart = cg.rows != cg.cols;
  return it;
}

// Persistent: one workgroup per CU (its table fills the LDS) takes items
// blockIdx.x, + gridDim.x, ...: the row planes of the next item and the first
// columns of this one are loaded while the table is cleared, filled and
// summed, which as a launch of one workgroup per item left the CU idle for
// 11 us of every 15 (1,501 samples) to 40 us (8,192).  The groups of one
// (k-mer length, half) run side by side, as they read the same columns; the
// grid has no common factor with the number of groups, so that every
// workgroup meets long and short ones alike.
__global__ __launch_bounds__(CODE_TB) void code_kernel(DistParams p, const CodeGroup* groups,
                                                       int n_groups, int n_items) {
  __shared__ uint2 tab[32 * 512];
  __shared__ uint32_t s_most;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  constexpr int HALF_TB = CODE_TB / 2;
  const int r = (int)(threadIdx.x & (HALF_TB - 1));
  const bool high = threadIdx.x >= HALF_TB;
  CodeItem it = code_item(p, groups, n_groups, (int)blockIdx.x);
  uint32_t rpl[BBITS];
  load_planes(code_source(it.rows, min(it.rows.s0 + r, it.rows.s1 - 1)), rpl);
  for (int item = (int)blockIdx.x; item < n_items; item += (int)gridDim.x) {
    uint32_t cpl[BBITS];
    load_planes(code_source(it.cols, min(it.cols.s0 + (int)threadIdx.x, it.cols.s1 - 1)), cpl);
    uint4* clr = reinterpret_cast<uint4*>(tab);
    for (int x = threadIdx.x; x < 32 * 512 / 2; x += CODE_TB) clr[x] = make_uint4(0, 0, 0, 0);
    if (threadIdx.x == 0) s_most = 0;
    __syncthreads();
    // rows into the bitmaps: lanes 0 .. 511 the low 16 bins of a row, the
    // others the high 16
    for (int row = it.rows.s0 + r; row < it.rows.s1; row += HALF_TB) {
      if (row >= it.rows.s0 + HALF_TB) load_planes(code_source(it.rows, row), rpl);
      uint32_t x[16];
      to_values(rpl, x);
      uint2* t = tab + (high ? 16 * 512 : 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t v = high ? x[i] >> 16 : x[i] & 0xFFFFu;
        atomicOr(&t[i * 512 + (v >> 5)].x, 0x80000000u >> (v & 31));
      }
    }
    __syncthreads();
    // ranks: each wave takes two bins, lane l the dwords l, 64 + l, ...; the
    // order of the dwords does not matter, only that every value's rank differs
    {
      uint2* t0 = tab + (wave * 2) * 512 + lane;
      uint2* t1 = t0 + 512;
      uint32_t n0[8], n1[8], sum0 = 0, sum1 = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        n0[i] = sum0;
        n1[i] = sum1;
        sum0 += __popc(t0[i * 64].x);
        sum1 += __popc(t1[i * 64].x);
      }
      const uint32_t incl0 = wave_prefix(sum0), incl1 = wave_prefix(sum1);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        t0[i * 64].y = incl0 - sum0 + n0[i];
        t1[i * 64].y = incl1 - sum1 + n1[i];
      }
      if (lane == 63) atomicMax(&s_most, max(incl0, incl1));
    }
    __syncthreads();
    const int width = max(3, 32 - __clz((int)s_most));
    if (threadIdx.x == 0) it.widths[it.kh] = (uint32_t)width;
    const CodeItem now = it;
    if (item + (int)gridDim.x < n_items) {
      it = code_item(p, groups, n_groups, item + (int)gridDim.x);
      load_planes(code_source(it.rows, min(it.rows.s0 + r, it.rows.s1 - 1)), rpl);
    }
    if (width <= 8) {
      code_samples<8>(now.cols, tab, width, cpl);
    } else {
      code_samples<16>(now.cols, tab, width, cpl);
    }
    if (now.apart) {
      load_planes(code_source(now.rows, min(now.rows.s0 + (int)threadIdx.x, now.rows.s1 - 1)), cpl);
      if (width <= 8) {
        code_samples<8>(now.rows, tab, width, cpl);
      } else {
        code_samples<16>(now.rows, tab, width, cpl);
      }
    }
    __syncthreads();  // the table is free
  }
}

// ---------------------------------------------------------------------------
// Matching of coded planes (dist_coded).  The same wave grid, operand pipeline
// and rules as match_stage_pipe; a half of width P is P planes in an even
// number of batches of 2 planes, then of 1 (so that the two register sets keep
// their roles); the first always has 2, so that the last batch of a half can
// issue the first of the next half whatever its width.  (Batches of 3 would
// make widths 5, 9 and 10 shorter, but their third row tuple spills SGPRs.)
// ---------------------------------------------------------------------------
constexpr int code_batches(int P) { return P <= 4 ? 2 : (P <= 8 ? 4 : 6); }
constexpr int code_batch(int P, int b) {  // planes of batch b: as many of 2 as leave 1 for the rest
  return b < P - code_batches(P) ? 2 : 1;
}
constexpr int code_first(int P, int b) { return b == 0 ? 0 : code_first(P, b - 1) + code_batch(P, b - 1); }
static_assert(code_first(3, 2) == 3 && code_first(4, 2) == 4 && code_first(5, 4) == 5 &&
                  code_first(6, 4) == 6 && code_first(7, 4) == 7 && code_first(8, 4) == 8 &&
                  code_first(9, 6) == 9 && code_first(10, 6) == 10,
              "batches cover the planes of every width");
static_assert(code_batch(3, 0) == 2 && code_batch(5, 0) == 2 && code_batch(9, 0) == 2,
              "the first batch has 2 planes");

// Operands of up to 2 planes: 8 rows in SGPRs and RR columns per lane each.
template <int RR>
struct CodeBatch {
  ATuple<8>::T a[2];
  u32x2 b[2][RR == 4 ? 2 : 1];
};

// Issue NP planes: row plane x at aw + AOFF + 1024 x bytes, column plane x at
// LDS address bw + (BP + x) KiB.
template <int RR, int NP, int AOFF, int BP>
__device__ __forceinline__ void code_issue(const CU32* aw, uint32_t bw, CodeBatch<RR>& x) {
  a_load<8, AOFF>(aw, x.a[0]);
  if constexpr (NP > 1) a_load<8, AOFF + 1024>(aw, x.a[1]);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    if constexpr (RR == 1) {
      asm volatile("ds_read_b32 %0, %1 offset:%2"
                   : "=&v"(x.b[i][0].x)
                   : "v"(bw), "i"((BP + i) * 1024));
    } else {
#pragma unroll
      for (int r = 0; r < RR / 2; ++r) {
        asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3"
                     : "=&v"(x.b[i][r])
                     : "v"(bw), "i"((BP + i) * 4 + 2 * r), "i"((BP + i) * 4 + 2 * r + 1));
      }
    }
  }
}

// WAIT: the wait for a batch's loads; else only keeps its registers alive and
// in place at this point (batch_hold).  Two asm blocks, as the compiler takes
// every output of a block that also has vector outputs for divergent and would
// move the row operands through VGPRs where paths join.
template <int RR, int NP, bool WAIT>
__device__ __forceinline__ void code_pin(CodeBatch<RR>& x) {
  if constexpr (WAIT && NP == 2) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(x.a[0]), "+s"(x.a[1]));
  } else if constexpr (WAIT) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(x.a[0]));
  } else if constexpr (NP == 2) {
    asm volatile("" : "+s"(x.a[0]), "+s"(x.a[1]));
  } else {
    asm volatile("" : "+s"(x.a[0]));
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    if constexpr (RR == 4) {
      asm volatile("" : "+v"(x.b[i][0]), "+v"(x.b[i][1]));
    } else if constexpr (RR == 2) {
      asm volatile("" : "+v"(x.b[i][0]));
    } else {
      asm volatile("" : "+v"(x.b[i][0].x));
    }
  }
}

// Batches B .. of one half of width P; cur holds batch B (complete).  The
// last one issues the first batch of the next half: its row planes lie one
// slot on, its column planes follow in the stage (past the stage's last half
// the loads read other bytes of the buffers, which nothing uses).
template <int RR, int P, int B>
__device__ __forceinline__ void code_match(const CU32* aw, uint32_t bw, CodeBatch<RR>& cur,
                                           CodeBatch<RR>& nxt, uint32_t (&acc)[8][RR],
                                           uint32_t (&cnt)[8][RR]) {
  constexpr int NB = code_batches(P), NP = code_batch(P, B), P0 = code_first(P, B);
  if constexpr (B + 1 < NB) {
    code_issue<RR, code_batch(P, B + 1), (P0 + NP) * 1024, P0 + NP>(aw, bw, nxt);
  } else {
    code_issue<RR, 2, CODE_SLOT * 4, P>(aw, bw, nxt);
  }
  code_pin<RR, NP, false>(cur);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        const uint32_t a = cur.a[i][q];
        const uint32_t b = cur.b[i][r / 2][r % 2];
        acc[q][r] = P0 + i == 0 ? ~(a ^ b) : match_and(acc[q][r], a, b);
      }
    }
  }
  if constexpr (B + 1 < NB) {
    code_pin<RR, code_batch(P, B + 1), true>(nxt);
    code_match<RR, P, B + 1>(aw, bw, nxt, cur, acc, cnt);
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        asm("v_bcnt_u32_b32 %0, %1, %0" : "+v"(cnt[q][r]) : "v"(acc[q][r]));
      }
    code_pin<RR, 2, true>(nxt);
  }
}

// The next halves of the stage as long as they are P planes wide (widths left
// in ws, 4 bits each).
template <int RR, int P>
__device__ __forceinline__ void code_halves(const CU32*& aw, uint32_t& bw, uint32_t& ws,
                                            CodeBatch<RR>& c, CodeBatch<RR>& n,
                                            uint32_t (&cnt)[8][RR]) {
  while ((ws & 15u) == (uint32_t)P) {
    uint32_t acc[8][RR];
    code_match<RR, P, 0>(aw, bw, c, n, acc, cnt);
    aw += CODE_SLOT;
    bw += P * 1024;
    ws >>= 4;
  }
}

// A stage: as many whole halves as fit CODE_STAGE planes, at most 8; widths
// packed 4 bits each.
struct CodeStage {
  uint32_t widths;
  int halves, planes;
};

typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ CodeStage code_stage(const u32x8& w, int left) {
  CodeStage st{0, 0, 0};
#pragma unroll
  for (int i = 0; i < 8; ++i) st.widths |= (w[i] & 15u) << (4 * i);
  st.widths = __builtin_amdgcn_readfirstlane(st.widths);
  const int most = left < 8 ? left : 8;
  while (st.halves < most) {
    const int planes = st.planes + (int)((st.widths >> (4 * st.halves)) & 15u);
    if (planes > CODE_STAGE) break;
    st.planes = planes;
    st.halves += 1;
  }
  if (st.halves < 8) st.widths &= (1u << (4 * st.halves)) - 1u;
  return st;
}

// Copies of one stage: column planes (1 KiB each, one wave instruction)
// packed into the stage buffer, plane l of a half by wave l % 8; row planes, 4 at a time
// (64 rows each), into a scratch KiB that nothing reads, only so that the
// scalar loads find them in L2.
__device__ __forceinline__ void code_copy(const CodeStage& st, const uint32_t* cols,
                                          const uint32_t* rows, bool rpf, uint32_t dst,
                                          uint32_t row_dst, int wave, uint32_t coff,
                                          uint32_t roff) {
  for (int x = 0; x < st.halves; ++x) {
    const int w = (int)(st.widths >> (4 * x)) & 15;
    if (wave < w) dma16<0>(cols + wave * 256, coff, dst + (uint32_t)wave * 1024);
    if (wave + WAVES < w) {
      dma16<WAVES * 1024>(cols + (wave + WAVES) * 256, coff, dst + (uint32_t)wave * 1024);
    }
    const int quad = (wave - 3 * x) & (WAVES - 1);  // quads 0 .. 2 of the half
    if (rpf && 4 * quad < w) dma16<0>(rows + quad * 1024, roff, row_dst);
    cols += CODE_SLOT;
    rows += CODE_SLOT;
    dst += (uint32_t)w * 1024;
  }
}

template <int RR>
__device__ __forceinline__ void coded_item(const CU32* widths, const uint32_t* cols,
                                           const uint32_t* rows, bool rpf, int halves,
                                           uint32_t buf, uint32_t row_dst, uint16_t* counts,
                                           int wave, int lane) {
  constexpr int CG = TileCfg<8, RR>::CG;
  const uint32_t coff = (uint32_t)lane * 16;
  const uint32_t roff = (uint32_t)((lane >> 4) * 1024 + (lane & 15) * 16);
  const uint32_t col = (uint32_t)((wave % CG) * 64 * RR + lane) * 4;
  const CU32* arow = (CU32*)(rows + (wave / CG) * 8);
  uint32_t cnt[8][RR];
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int r = 0; r < RR; ++r) cnt[q][r] = 0;
  CodeBatch<RR> c, n;
  u32x8 w8;
  asm volatile("s_load_dwordx8 %0, %1, 0\n\ts_waitcnt lgkmcnt(0)" : "=&s"(w8) : "s"(widths));
  CodeStage cur = code_stage(w8, halves);
  code_copy(cur, cols, rows, rpf, buf, row_dst, wave, coff, roff);
  int h = 0;  // first half of the current stage
  uint32_t at = buf;
  asm volatile("s_load_dwordx8 %0, %1, 0\n\ts_waitcnt lgkmcnt(0)"
               : "=&s"(w8)
               : "s"(widths + cur.halves));
  CodeStage nxt = code_stage(w8, halves - cur.halves);
  for (;;) {
    // one barrier per stage, as in tile_stages
    wait_vmcnt<0>();
    stage_barrier();
    const int h1 = h + cur.halves;
    const uint32_t other = buf + (at == buf ? (uint32_t)CODE_STAGE * 1024 : 0u);
    code_copy(nxt, cols + (int64_t)h1 * CODE_SLOT, rows + (int64_t)h1 * CODE_SLOT, rpf, other,
              row_dst, wave, coff, roff);
    const CU32* aw = arow + (int64_t)h * CODE_SLOT;
    uint32_t bw = at + col;
    code_issue<RR, 2, 0, 0>(aw, bw, c);
    // the widths of the stage after the next arrive with the first batch
    asm volatile("s_load_dwordx8 %0, %1, 0\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(w8)
                 : "s"(widths + h1 + nxt.halves));
    code_pin<RR, 2, true>(c);
    const CodeStage after = code_stage(w8, halves - h1 - nxt.halves);
    // one loop per width, in turn until the stage is done: a value has one
    // successor at every step, so the counts and operands stay in their
    // registers (a switch moves all of them at every half: 44 moves beside the
    // 288 operations of 8 planes)
    uint32_t ws = cur.widths;
    while (ws != 0) {
      code_halves<RR, 8>(aw, bw, ws, c, n, cnt);
      code_halves<RR, 7>(aw, bw, ws, c, n, cnt);
      code_halves<RR, 6>(aw, bw, ws, c, n, cnt);
      code_halves<RR, 9>(aw, bw, ws, c, n, cnt);
      code_halves<RR, 5>(aw, bw, ws, c, n, cnt);
      code_halves<RR, 4>(aw, bw, ws, c, n, cnt);
      code_halves<RR, 3>(aw, bw, ws, c, n, cnt);
      code_halves<RR, 10>(aw, bw, ws, c, n, cnt);
    }
    if (nxt.halves == 0) break;
    h = h1;
    cur = nxt;
    nxt = after;
    at = other;
  }
  store_counts<8, RR>(counts, 0, wave, lane, cnt);
}

__global__ __launch_bounds__(WAVES * 64, 4) void dist_coded(DistParams p, ItemArgs a,
                                                            const CodeGroup* groups) {
  // two stages; the row scratch KiB, and what the last operand batch of a stage
  // reads past it (2 planes)
  __shared__ uint4 s_buf[2 * CODE_STAGE * 64 + 3 * 64];
  __shared__ int s_stop;
  const int all = 2 * p.s64;  // halves of a sketch
  ItemAt it;
  if (!item_at(a, p.n_k, all, it)) return;
  if (p.ctl.stop != nullptr && blockIdx.x >= (uint32_t)a.unwatched) {
    if (threadIdx.x == 0) s_stop = item_stopped(p.ctl, blockIdx.x) ? 1 : 0;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_stop)) return;
  }
  const int kk = it.kk;
  const ItemTile tile = a.tiles[it.tile];
  const int row0 = __builtin_amdgcn_readfirstlane(tile.row0);
  const int ct = __builtin_amdgcn_readfirstlane(tile.ct);
  const int rows = __builtin_amdgcn_readfirstlane(tile.rows);
  // scalar loads: the table is never written while the kernel runs
  CCodeGroup& g = ((CCodeGroup*)groups)[__builtin_amdgcn_readfirstlane(tile.group)];
  const int h0 = it.unit0;
  const int halves = it.units;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t block = (int64_t)all * CODE_SLOT;
  const int64_t at = (int64_t)h0 * CODE_SLOT;
  const uint32_t* cols = g.cols + ((int64_t)kk * g.ncb + (ct - g.cb0)) * block + at;
  const uint32_t* rws =
      g.rows + ((int64_t)kk * g.nrb + (row0 / 256 - g.rb0)) * block + at + row0 % 256;
  const CU32* widths = (CU32*)(g.widths + kk * all + h0);
  uint16_t* counts = p.counts + it.block * ITEM_COUNTS;
  const uint32_t buf = lds_addr(s_buf);
  const uint32_t row_dst = buf + 2 * CODE_STAGE * 1024;
  const bool rpf = p.row_prefetch != 0;
  if (rows == 64) {
    coded_item<4>(widths, cols, rws, rpf, halves, buf, row_dst, counts, wave, lane);
  } else if (rows == 32) {
    coded_item<2>(widths, cols, rws, rpf, halves, buf, row_dst, counts, wave, lane);
  } else {
    coded_item<1>(widths, cols, rws, rpf, halves, buf, row_dst, counts, wave, lane);
  }
  if (threadIdx.x == 0) add_item(p.ctl);
}

hipError_t launch_coded(const DistParams& p, const ItemArgs& a, const CodeGroup* groups,
                        int first_group, int n_groups, hipStream_t stream) {
  if (a.n_items <= 0 || n_groups <= 0) return hipSuccess;
  const int n_code = n_groups * p.n_k * 2 * p.s64;
  int dev = 0, grid = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&grid, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  while (grid > 1 && std::gcd(grid, n_groups) != 1) --grid;
  code_kernel<<<(unsigned)std::min(grid, n_code), CODE_TB, 0, stream>>>(p, groups + first_group,
                                                                        n_groups, n_code);
  // never the matching of planes that were not coded: it walks their widths
  if ((e = hipGetLastError()) != hipSuccess) return e;
  dist_coded<<<item_grid(a), WAVES * 64, 0, stream>>>(p, a, groups);
  dist_items_out<<<(unsigned)(a.n_tiles * (64 / a.out_rows)), 256, 0, stream>>>(p, a);
  return hipGetLastError();
}

__global__ void batch_reset_kernel(uint32_t* queue_next, unsigned long long* fail, int n_jobs,
                                   unsigned long long* progress) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x < BATCH_QUEUES) queue_next[x] = 0u;
  if (x == 0 && progress) *progress = 0ull;
  if (fail && x < n_jobs) {
    fail[2 * x] = 0ull;
    fail[2 * x + 1] = ~0ull;
  }
}

__global__ void band_setup_kernel(ItemTile* tiles, int64_t rows, BandTiles b, int64_t n_ct, int64_t step,
                                  unsigned long long* fail, uint32_t* fail_rows) {
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x < rows) fail_rows[x] = 0u;
  if (x == 0) {
    fail[0] = 0ull;
    fail[1] = ~0ull;
  }
  if (step == 0) return;
  const int64_t per = b.tall + b.shorts;  // tiles of a column block
  if (x >= per * n_ct) return;
  const int64_t c0 = x / (per * step) * step;
  const int64_t nc = n_ct - c0 < step ? n_ct - c0 : step;
  const int64_t y = x - c0 * per;
  if (y < nc * b.tall) {
    tiles[x] = {(int32_t)(y % b.tall * 64), (int32_t)(c0 + y / b.tall), 64, 0};
  } else {
    const int64_t z = y - nc * b.tall;
    const int second = (int)(z % b.shorts);
    tiles[x] = {(int32_t)(b.tall * 64 + second * b.first), (int32_t)(c0 + z / b.shorts),
                second ? 16 : b.first, 0};
  }
}

hipError_t launch_band_setup(ItemTile* tiles, int64_t rows, const BandTiles& b, int64_t n_ct, int64_t step,
                             unsigned long long* fail, uint32_t* fail_rows, hipStream_t stream) {
  int64_t n = rows > 0 ? rows : 1;
  if (step > 0 && (b.tall + b.shorts) * n_ct > n) n = (b.tall + b.shorts) * n_ct;
  band_setup_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(tiles, rows, b, n_ct, step, fail,
                                                                     fail_rows);
  return hipGetLastError();
}

__global__ void call_reset_kernel(unsigned long long* fail, Control ctl) {
  fail[0] = 0ull;
  fail[1] = ~0ull;
  *ctl.progress = 0ull;
  *ctl.stop = 0u;
}

hipError_t launch_call_reset(unsigned long long* fail, const Control& ctl, hipStream_t stream) {
  call_reset_kernel<<<1, 1, 0, stream>>>(fail, ctl);
  return hipGetLastError();
}

bool variant_valid(int v) { return v >= 1 && v <= N_VARIANTS; }

int variant_tile_rows(int v) {
  switch (v) {
    case 1:
    case 3:
      return 128;
    case 4:
      return 32;
    case 5:
      return 16;
    default:
      return 64;
  }
}

int variant_tile_cols(int v) {
  switch (v) {
    case 1:
      return 64;
    case 3:
      return 128;
    default:
      return 256;
  }
}

hipError_t launch_dists(const DistParams& p, int variant, int64_t n_items, hipStream_t stream) {
  if (n_items <= 0) return hipSuccess;
  const unsigned g = (unsigned)n_items;
  switch (variant) {
    case 1:
      dist_tiles<16, 1, 0><<<g, WAVES * 64, 0, stream>>>(p);
      break;
    case 3:
      dist_tiles<16, 2, 0><<<g, WAVES * 64, 0, stream>>>(p);
      break;
    case 4:
      dist_tiles<8, 2, 2><<<g, WAVES * 64, 0, stream>>>(p);
      break;
    case 5:
      dist_tiles<8, 1, 2><<<g, WAVES * 64, 0, stream>>>(p);
      break;
    default:
      dist_tiles<8, 4, 2><<<g, WAVES * 64, 0, stream>>>(p);
      break;
  }
  return hipGetLastError();
}

// Batch kernels exist for the pipelined shapes only; BATCH_MIXED runs the
// shape each item names.
template <typename F>
static hipError_t with_batch_kernel(int variant, F f) {
  switch (variant) {
    case 4:
      return f(dist_batch<8, 2, 2>);
    case 2:
      return f(dist_batch<8, 4, 2>);
    case BATCH_MIXED:
      return f(dist_batch_mixed);
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t batch_grid(int variant, int* grid) {
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  return with_batch_kernel(variant, [&](auto kern) {
    int per_cu = 0;
    hipError_t r = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, WAVES * 64, 0);
    if (r != hipSuccess) return r;
    *grid = (per_cu > 0 ? per_cu : 1) * cus;
    return hipSuccess;
  });
}

hipError_t launch_batch(const BatchArgs& a, int variant, int grid, hipStream_t stream) {
  if (grid <= 0) return hipErrorInvalidValue;
  return with_batch_kernel(variant, [&](auto kern) {
    kern<<<grid, WAVES * 64, 0, stream>>>(a);
    return hipGetLastError();
  });
}

hipError_t launch_batch_reset(uint32_t* queue_next, unsigned long long* fail, int n_jobs,
                              hipStream_t stream, unsigned long long* progress) {
  const int n = n_jobs > BATCH_QUEUES ? n_jobs : BATCH_QUEUES;
  batch_reset_kernel<<<(n + 255) / 256, 256, 0, stream>>>(queue_next, fail, n_jobs, progress);
  return hipGetLastError();
}

__global__ void tile_reset_kernel(uint32_t* tile_done, int64_t n, unsigned long long* fail) {
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x < n) tile_done[x] = 0u;
  if (x == 0 && fail) {
    fail[0] = 0ull;
    fail[1] = ~0ull;
  }
}

hipError_t launch_dists_diagonal(const DistParams& p, int64_t n_items, hipStream_t stream) {
  if (n_items <= 0) return hipSuccess;
  dist_tiles_diagonal<<<(unsigned)n_items, WAVES * 64, 0, stream>>>(p);
  return hipGetLastError();
}

hipError_t upload_log_table() {
  double tab[LOG_TAB_DOUBLES];
  log_table_fill(tab);
  return hipMemcpyToSymbol(HIP_SYMBOL(g_log_tab), tab, sizeof(tab));
}

hipError_t launch_tile_reset(uint32_t* tile_done, int64_t n, unsigned long long* fail,
                             hipStream_t stream) {
  const int64_t m = n > 1 ? n : 1;
  tile_reset_kernel<<<(unsigned)((m + 255) / 256), 256, 0, stream>>>(tile_done, n, fail);
  return hipGetLastError();
}

}  // namespace ppsk
