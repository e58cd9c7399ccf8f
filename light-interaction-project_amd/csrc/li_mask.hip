// Block-mask builder for gfx950: pooled block similarity, forced AR blocks,
// per-query-block top-k and ascending block lists.
//
// Replaces fast_generate_indices (hy-worldplay/.../ar_sparse_operation.py:223-284)
// and generate_prefill_indices (bi_sparse_operation_for_KV_cache.py:220-296,
// matrix-game-3.0/.../bi_sparse_operation.py:179-234), which run normalize /
// matmul / +1e6 bias / topk / sort / cat as a chain of torch launches.  Here one
// 256-thread workgroup per (query block, batch*head) does all of it:
//
// 1. score[j] for every key block j, with the reference's rounding points:
//    cosine  xn = E(x / max(E(sqrt(sum x^2)), E(1e-12))), sim = E(sum qn*kn);
//    scaled  sim = E(f32(E(sum q*k)) * scale);  dot  sim = E(sum q*k)
//    (E = round to the element type).  Element products are exact in fp32.
//    A dot product over d takes eight fp32 partial sums, partial i over
//    d = i, i+8, ... sequentially from +0.0, combined as
//    ((s0+s1)+(s2+s3))+((s4+s5)+(s6+s7)) (eight short chains instead of one
//    of D dependent multiply-adds); a sum of squares runs sequentially.
// 2. forced blocks (recent slabs, diagonal, sink, 3D neighbours) are kept
//    unconditionally -- the reference's +1e6 bias has the same effect;
// 3. the budget k follows the reference's integer arithmetic (int() truncation
//    of a double product) and the remaining k - n_forced blocks are the
//    largest non-forced scores, ties to the lower index: every key block gets
//    the unique 32-bit key (order-preserving score bits << 16 | 0xFFFF - j;
//    0 marks a forced block) and a search two bits at a time finds a
//    threshold with exactly k - n_forced non-forced keys at or above it;
// 4. the selected blocks are written in ascending order by a ballot/prefix
//    compaction over j, which replaces the reference's topk + sort.
//
// One wave selects each query row: every per-row reduction is a ballot +
// popcount inside that wave, and the row's 32-bit keys live in LDS (4 bytes
// per key block).  Aligned pools with a unit d stride take the shared-pool
// kernel (4 rows of one head per workgroup, each wave scoring every fourth or
// eighth chunk of 64 blocks against all of them); other pools and very long key
// grids take the generic kernel, in which each wave scores its row by reading
// the pool rows itself.
#include "li_common.hpp"

namespace li {
namespace {

constexpr int kMaxNk = 12288;

struct MaskArgs {
  const uint16_t* qp;
  int64_t qs[4];
  const uint16_t* kp;
  int64_t ks[4];
  li_mask_params p;
  int32_t* indices;
  int32_t* counts;
  uint16_t* scores;
  int32_t NH, NBH, groups;  // heads, batch * heads, row groups of a head (shared-pool path)
  uint32_t mg_hw, mg_nw;  // udiv16 magics of nh nw and nw (0 for 1 and past 2^16, where no block lies)
};

__device__ __forceinline__ uint32_t order16(uint16_t bits) {
  return (bits & 0x8000u) ? (uint32_t)(~bits & 0xFFFFu) : (uint32_t)(bits | 0x8000u);
}

template <typename E, int D>
__device__ __forceinline__ void load_row(const uint16_t* p, int64_t stride, bool vec, float* x) {
  if (vec) {
#pragma unroll
    for (int c = 0; c < D / 8; ++c) {
      u32x4 w = *reinterpret_cast<const u32x4*>(p + 8 * c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[8 * c + 2 * i] = E::to_f32(uint16_t(w[i] & 0xFFFFu));
        x[8 * c + 2 * i + 1] = E::to_f32(uint16_t(w[i] >> 16));
      }
    }
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = E::to_f32(p[d * stride]);
  }
}

// Sequential fp32 sum of squares from +0.0, then the reference's normaliser
// max(E(sqrt(.)), E(1e-12)).
template <typename E, int D>
__device__ __forceinline__ float norm_den(const float* x) {
  float ss = 0.0f;
#pragma unroll
  for (int d = 0; d < D; ++d) ss = ss + x[d] * x[d];
  const float nrm = E::to_f32(E::from_f32(__builtin_sqrtf(ss)));
  const float eps = E::to_f32(E::from_f32(1e-12f));
  return nrm > eps ? nrm : eps;
}

__device__ __forceinline__ int wave_count(bool pred) { return __popcll(__ballot(pred)); }

// The dot product's combination of its eight partial sums.
__device__ __forceinline__ float sum8(const float* s) {
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

#define LI_SEL_INLINE __attribute__((always_inline))

// Steps 3 and 4 for query row qb of (b, h) = bh, run by one wave: key_at(r)
// is the key of block 64 r + lane (0 for forced blocks and past nk), nchunk =
// ceil(nk / 64), nf the number of forced blocks.
template <int KUNROLL, typename KeyAt>
__device__ __forceinline__ void select_row(const MaskArgs& a, KeyAt&& key_at, int nchunk, int nf, int qb, int bh,
                                           int lane) {
  const li_mask_params& p = a.p;
  const int nk = p.nk;

  // 3. budget.
  int k;
  if (p.row_budget) {
    k = p.row_budget[qb];
    k = k < nf ? nf : k;
    k = k > nk ? nk : k;
  } else if (p.budget_mode == LI_BUDGET_HISTORY) {
    k = nf + (int)((double)(nk - nf) * p.topk_ratio);
    const int lo = nk > 0 ? 1 : 0;
    k = k < lo ? lo : k;
    k = k > nk ? nk : k;
    k = k < nf ? nf : k;
  } else {
    k = (int)((double)nk * p.topk_ratio);
    k = k < p.min_budget ? p.min_budget : k;
    k = k > nk ? nk : k;
    k = k < nf ? nf : k;
  }
  // Wave-uniform, so the search below runs on scalar registers.
  const int kk = __builtin_amdgcn_readfirstlane(k - nf);  // non-forced blocks to keep
  const int nfree = nk - nf;

  // Threshold thr with exactly kk non-forced keys >= thr, found from the top
  // two bits per step: with the bits above settled in `prefix`, the three
  // candidates prefix|11, prefix|10 and prefix|01 are counted together (their
  // ballots are independent), and the largest one with at least kk keys at
  // or above it is kept -- what two single-bit steps would keep.  Forced keys
  // are 0 and never reach a candidate, which is always >= 1 here.  The search
  // stops as soon as a kept candidate has exactly kk keys at or above it, the
  // same set as the kk-th largest key selects; for distinct scores that
  // happens within the 16 score bits.  Index bits 15 .. L-1 of the low half
  // are 1 in every key (0xFFFF - j with j < nk <= 2^L): they are set in the
  // prefix from the start (no key's count changes) and not searched.
  uint32_t thr = 1u;
  if (kk > 0 && kk < nfree) {
    const int L = nk > 1 ? 32 - __builtin_clz((uint32_t)(nk - 1)) : 0;
    // The searched bit below b, or -1.
    auto below = [&](int b) LI_SEL_INLINE { return b - 1 >= 16 || b - 1 < L ? b - 1 : L - 1; };
    uint32_t prefix = 0xFFFFu & ~((1u << L) - 1u);
    int b1 = 31;
    if constexpr (KUNROLL > 4) {
      // Many keys per lane: the counts cost more than the steps' latency, and
      // one candidate per bit counts a third less than three per two bits.
      for (; b1 >= 0; b1 = below(b1)) {
        const uint32_t c = prefix | (1u << b1);
        int n = 0;
#pragma unroll KUNROLL
        for (int r = 0; r < nchunk; ++r) n += wave_count(key_at(r) >= c);
        if (n >= kk) {
          prefix = c;
          if (n == kk) break;
        }
      }
      b1 = -1;
    }
    while (b1 >= 0) {
      const int b0 = below(b1);
      const uint32_t m1 = 1u << b1, m0 = b0 >= 0 ? 1u << b0 : 0u;
      const uint32_t c3 = prefix | m1 | m0, c2 = prefix | m1, c1 = prefix | m0;
      int n3 = 0, n2 = 0, n1 = 0;
#pragma unroll KUNROLL
      for (int r = 0; r < nchunk; ++r) {
        const uint32_t key = key_at(r);
        n3 += wave_count(key >= c3);
        n2 += wave_count(key >= c2);
        n1 += wave_count(key >= c1);
      }
      if (n3 >= kk) {
        prefix = c3;
        if (n3 == kk) break;
      } else if (n2 >= kk) {
        prefix = c2;
        if (n2 == kk) break;
      } else if (m0 != 0u && n1 >= kk) {
        prefix = c1;
        if (n1 == kk) break;
      }
      b1 = b0 >= 0 ? below(b0) : -1;
    }
    thr = prefix;
  }

  // 4. ascending compaction.
  const int64_t row = (int64_t)bh * p.nq + qb;
  int32_t* irow = a.indices + row * p.kmax;
  const int ntxt = p.num_txt_blk;
  for (int i = lane; i < ntxt && i < p.kmax; i += 64) irow[i] = i;
  int base = ntxt;
#pragma unroll KUNROLL
  for (int r = 0; r < nchunk; ++r) {
    const int j = r * 64 + lane;
    bool sel = false;
    if (j < nk) {
      const uint32_t key = key_at(r);
      sel = key == 0u || (kk > 0 && key >= thr);
    }
    const uint64_t m = __ballot(sel);
    const int dst = base + __popcll(m & ((1ull << lane) - 1ull));
    if (sel && dst < p.kmax) irow[dst] = j + ntxt;
    base += __popcll(m);
  }
  for (int i = ntxt + k + lane; i < p.kmax; i += 64) irow[i] = 0;
  if (lane == 0) a.counts[row] = ntxt + k;
}

#define LI_MASK_INLINE __attribute__((always_inline))

// Query row qb of (b, h) into qv (fp32, D values), normalised for cosine: every
// lane computes the same sequential normaliser; lanes own d = lane, lane + 64, ...
template <typename E, int D>
__device__ __forceinline__ void load_query(const MaskArgs& a, int b, int h, int qb, bool cosine, float* qv,
                                           int lane) {
  const uint16_t* qrow = a.qp + b * a.qs[0] + h * a.qs[1] + (int64_t)qb * a.qs[2];
  // All of the lane's loads are issued before the first is used.
  constexpr int PER = (D + 63) / 64;
  uint16_t x[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int d = lane + 64 * i;
    x[i] = d < D ? qrow[(int64_t)d * a.qs[3]] : uint16_t(0);
  }
#pragma unroll
  for (int i = 0; i < PER; ++i)
    if (lane + 64 * i < D) qv[lane + 64 * i] = E::to_f32(x[i]);
  __builtin_amdgcn_wave_barrier();
  if (cosine) {
    float ss = 0.0f;
    for (int d = 0; d < D; ++d) ss = ss + qv[d] * qv[d];
    const float nrm = E::to_f32(E::from_f32(__builtin_sqrtf(ss)));
    const float eps = E::to_f32(E::from_f32(1e-12f));
    const float den = nrm > eps ? nrm : eps;
    __builtin_amdgcn_wave_barrier();
    for (int d = lane; d < D; d += 64) qv[d] = E::to_f32(E::from_f32(qv[d] / den));
    __builtin_amdgcn_wave_barrier();
  }
}

// A query row's position in the key grid, for the forced-block tests.
struct RowGeom {
  int nk, qb, pos, hw, sink, pt, ph, pw;
  __device__ RowGeom(const li_mask_params& p, int qb_, uint32_t mg_hw, uint32_t mg_nw) : nk(p.nk), qb(qb_) {
    pos = p.nk - p.nq + qb;  // query block's position in the key grid
    hw = p.nh * p.nw;
    sink = qb < 65536 ? qb - (int)udiv16(qb, mg_hw) * hw : qb % hw;
    // Used for positions inside the key grid only (below 2^16).
    pt = (int)udiv16(pos, mg_hw);
    const int pr = pos - pt * hw;
    ph = (int)udiv16(pr, mg_nw);
    pw = pr - ph * p.nw;
  }
};

// Step 1b/2 for one (row, block): score bits from the dot product in E, the
// forced flag, and the order key (0 for a forced block).  mg_hw, mg_nw: udiv16
// magics of the key grid's slab and row (nk <= kMaxNk < 2^16).
template <typename E>
__device__ __forceinline__ uint32_t finish_key(const li_mask_params& p, const RowGeom& g, uint16_t* srow, int j,
                                               uint16_t s, bool& f, uint32_t mg_hw, uint32_t mg_nw) {
  if (p.metric == LI_METRIC_SCALED_DOT) s = E::from_f32(E::to_f32(s) * p.scale);
  if (srow) srow[j] = s;
  f = (p.n_recent > 0) && (j >= g.nk - p.n_recent);
  if (p.force_diag && j == g.pos) f = true;
  if (p.force_sink && j == g.sink) f = true;
  if (p.force_neighbors && g.pos >= 0 && g.pos < g.nk) {
    const int jt = (int)udiv16(j, mg_hw), jr = j - jt * g.hw, jh = (int)udiv16(jr, mg_nw), jw = jr - jh * p.nw;
    if (abs(jt - g.pt) + abs(jh - g.ph) + abs(jw - g.pw) <= 1) f = true;
  }
  return f ? 0u : ((order16(s) << 16) | (0xFFFFu - (uint32_t)j));
}

// Generic path (any pool strides, any nk <= kMaxNk): one wave per query row,
// `waves` rows per workgroup, each wave reading its head's pool rows itself;
// the keys live in the wave's LDS slice (nk + D words).
template <typename E, int D>
__global__ __launch_bounds__(256) void block_mask_kernel(MaskArgs a, int waves) {
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  const li_mask_params& p = a.p;
  const int nk = p.nk;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qb = blockIdx.x * waves + wave;
  const int bh = blockIdx.y;
  if (qb >= p.nq) return;  // whole wave leaves; no workgroup barrier follows
  const int b = bh / a.NH, h = bh % a.NH;
  const bool cosine = p.metric == LI_METRIC_COSINE;
  uint32_t* keys = smem + (size_t)wave * (nk + D);
  float* qv = reinterpret_cast<float*>(keys + nk);
  load_query<E, D>(a, b, h, qb, cosine, qv, lane);

  const RowGeom g(p, qb, a.mg_hw, a.mg_nw);
  const bool vec = a.ks[3] == 1 && (reinterpret_cast<uintptr_t>(a.kp) & 15u) == 0 && a.ks[0] % 8 == 0 &&
                   a.ks[1] % 8 == 0 && a.ks[2] % 8 == 0;
  const uint16_t* kbase = a.kp + b * a.ks[0] + h * a.ks[1];
  uint16_t* srow = a.scores ? a.scores + ((int64_t)bh * p.nq + qb) * nk : nullptr;
  int nf = 0;
  for (int j0 = 0; j0 < nk; j0 += 64) {
    const int j = j0 + lane;
    bool f = false;
    if (j < nk) {
      float x[D];
      load_row<E, D>(kbase + (int64_t)j * a.ks[2], a.ks[3], vec, x);
      float ps[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      if (cosine && !p.k_normalized) {
        const float den = norm_den<E, D>(x);
#pragma unroll
        for (int d = 0; d < D; ++d) ps[d & 7] = ps[d & 7] + qv[d] * E::to_f32(E::from_f32(x[d] / den));
      } else {
#pragma unroll
        for (int d = 0; d < D; ++d) ps[d & 7] = ps[d & 7] + qv[d] * x[d];
      }
      keys[j] = finish_key<E>(p, g, srow, j, E::from_f32(sum8(ps)), f, a.mg_hw, a.mg_nw);
    }
    nf += wave_count(f);
  }
  __builtin_amdgcn_wave_barrier();
  auto key_at = [&](int r) LI_MASK_INLINE {
    const int j = r * 64 + lane;
    return j < nk ? keys[j] : 0u;
  };
  select_row<1>(a, key_at, (nk + 63) / 64, nf, qb, bh, lane);
}

// Shared-pool path (16-byte aligned pools with unit d stride): a workgroup of
// eight waves holds 4 query rows of one (b, h).  Waves 0-3 load and normalise a
// query row each, while waves 4-7 stage the first chunks of 64 key blocks; SW
// waves (4-7, then for long grids 0-3 too) score a chunk each against all four
// rows, and waves 0-3 then finish and select a row each with the row's keys in
// registers (nk <= 64 KS).
//
// The kernel is a chain of latencies (one round of workgroups at most sizes), so
// the scoring is arranged to be short: a wave stages its chunk itself, straight
// to LDS, a lane converts its block's row once for all four query rows, and the
// products run on the matrix cores in fp32 (v_mfma_f32_4x4x1_16b_f32: sixteen
// 4 x 4 outer products, block by query row, for one d).  One such step adds one
// exact product to each sum and rounds once, as the generic path's multiply-add
// does, so partial sum i over d = i, i + 8, ... has the same bits.
// Kernel times, us, against one tile of 128 blocks at a time for the whole
// workgroup with two waves per row on the vector ALU (rows x blocks):
//   896 x 168  10.3 -> 9.9    1248 x 104 (cosine) 15.3 -> 11.4   256 x 64 (D = 64) 6.3 -> 6.1
//   2496 x 156 24.0 -> 16.6    720 x 150 (cosine) 11.7 -> 10.5   896 x 896 27.6 -> 25.6
// The scores wait for their selection in 16 bits (the type that they are rounded
// to first thing), which with SW = 4 leaves LDS for two workgroups a CU up to
// 1024 blocks; see li_block_mask for the choice of SW.
template <typename E, int D, int KS, int SW>
__global__ __launch_bounds__(512) void block_mask_rows_kernel(MaskArgs a) {
  constexpr int CH = D / 8;           // 16-byte granules per pool row
  constexpr int RB = 2 * D;           // bytes per pool row
  constexpr int RPI = 1024 / RB;      // rows per load instruction
  constexpr int QP = D + 4;           // query row pitch: the four rows in distinct banks
  typedef __attribute__((address_space(3))) void lds_void;
  __shared__ __attribute__((aligned(16))) char stage[SW][64 * RB];
  __shared__ __attribute__((aligned(16))) float qall[4][QP];
  __shared__ __attribute__((aligned(16))) uint16_t dots[4][64 * KS];
  // With a chunk per scoring wave at most, all waves share the raw pool's divisions.
  constexpr bool kShareDiv = KS <= SW;
  __shared__ float dens[kShareDiv ? 64 * KS : 1];
  const li_mask_params& p = a.p;
  const int nk = p.nk, nchunk = (nk + 63) / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup ids are dealt round-robin over the 8 XCDs; a contiguous range of
  // (head, row group) each lets the row groups of a head share one L2's copy of
  // its pool.
  const int n = a.groups * a.NBH, per = n >> 3, rem = n & 7, xcd = blockIdx.x & 7;
  const int pos = xcd * per + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
  const int bh = pos / a.groups, b = bh / a.NH, h = bh % a.NH;
  const int qb0 = (pos - bh * a.groups) * 4;
  const bool cosine = p.metric == LI_METRIC_COSINE;
  const uint16_t* kbase = a.kp + b * a.ks[0] + h * a.ks[1];
  const int sw = (wave + 4) & 7;  // scoring wave number: waves 4-7 first
  char* st = stage[sw < SW ? sw : 0];

  // Stage rows of 2 D bytes, granule g of row r at slot g ^ swz(r): the 16 lanes
  // that read granule c of 16 consecutive rows together then hit 16 distinct
  // windows.  Rows past nk repeat the last one; their keys are dropped.
  auto swz = [](int r) LI_MASK_INLINE { return D == 128 ? r & 15 : (r >> 1) & 7; };
  auto stage_chunk = [&](int chunk) LI_MASK_INLINE {
    const uint16_t* base = kbase + (int64_t)(64 * chunk) * a.ks[2];
    const uint32_t rstride = (uint32_t)(2 * a.ks[2]);
    const int last = nk - 1 - 64 * chunk;
    const uint32_t lds = (uint32_t)(uintptr_t)(lds_void*)st;
    const int r0 = lane / CH, slot = lane % CH;
#pragma unroll
    for (int n = 0; n < 64 / RPI; ++n) {
      const int r = n * RPI + r0;
      const uint32_t off = (uint32_t)(r < last ? r : last) * rstride + 16u * (slot ^ swz(r));
      dma16(base, off, lds + 1024 * n);
    }
  };
  const bool scores = sw < SW;
  if (wave >= 4 && sw < nchunk) stage_chunk(sw);
  // Rows past nq repeat the last one and are not selected.
  if (wave < 4) load_query<E, D>(a, b, h, qb0 + wave < p.nq ? qb0 + wave : p.nq - 1, cosine, qall[wave], lane);
  if (wave < 4 && scores && sw < nchunk) stage_chunk(sw);
  wait_vm0();
  __syncthreads();

  // Normaliser of this lane's block in the wave's stage, and the division of a
  // granule of a raw pool row by its normaliser.
  auto normaliser = [&]() LI_MASK_INLINE {
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(st + lane * RB + 16 * (c ^ swz(lane)));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = E::to_f32(uint16_t((w[i >> 1] >> (16 * (i & 1))) & 0xFFFFu));
        ss = ss + x * x;
      }
    }
    const float nrm = E::to_f32(E::from_f32(__builtin_sqrtf(ss)));
    const float eps = E::to_f32(E::from_f32(1e-12f));
    return nrm > eps ? nrm : eps;
  };
  auto divide = [&](char* at, float den) LI_MASK_INLINE {
    u32x4 w = *reinterpret_cast<u32x4*>(at);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t lo = E::from_f32(E::to_f32(uint16_t(w[e] & 0xFFFFu)) / den);
      const uint32_t hi = E::from_f32(E::to_f32(uint16_t(w[e] >> 16)) / den);
      w[e] = lo | (hi << 16);
    }
    *reinterpret_cast<u32x4*>(at) = w;
  };
  const bool raw_cosine = cosine && !p.k_normalized;
  if constexpr (kShareDiv) {
    if (raw_cosine) {
      if (scores && sw < nchunk) dens[64 * sw + lane] = normaliser();
      __syncthreads();
      // Granules of the rows that are there, eight divisions each: the longest part
      // of a small raw cosine call when a lane does its whole row (1 x 4 x 16 blocks,
      // D = 64: 6.8 us).
      for (int i = tid; i < nk * CH; i += 512) divide(stage[i / (64 * CH)] + (i % (64 * CH)) * 16, dens[i / CH]);
      __syncthreads();
    }
  }

  // Lane l of a 4x4x1 product: A = block l, B = query row l % 4; its result
  // element r is block 4 (l / 4) + r for query row l % 4.
  const float* qrow = qall[lane & 3];
  for (int chunk = scores ? sw : nchunk; chunk < nchunk; chunk += SW) {
    if (chunk != sw) wait_vm0();
    if (!kShareDiv && raw_cosine) {
      // The raw pool's rows, normalised in place by their lanes.
      const float den = normaliser();
#pragma unroll
      for (int c = 0; c < CH; ++c) divide(st + lane * RB + 16 * (c ^ swz(lane)), den);
    }
    f32x4 ps[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) ps[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(st + lane * RB + 16 * (c ^ swz(lane)));
      const f32x4 q0 = *reinterpret_cast<const f32x4*>(qrow + 8 * c);
      const f32x4 q1 = *reinterpret_cast<const f32x4*>(qrow + 8 * c + 4);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float k = E::to_f32(uint16_t((w[i >> 1] >> (16 * (i & 1))) & 0xFFFFu));
        ps[i] = __builtin_amdgcn_mfma_f32_4x4x1f32(k, i < 4 ? q0[i & 3] : q1[i & 3], ps[i], 0, 0, 0);
      }
    }
    // Every read of the stage has completed (its values went into the products).
    if (chunk + SW < nchunk) stage_chunk(chunk + SW);
    uint16_t dot[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float s8[8] = {ps[0][r], ps[1][r], ps[2][r], ps[3][r], ps[4][r], ps[5][r], ps[6][r], ps[7][r]};
      dot[r] = E::from_f32(sum8(s8));
    }
    *reinterpret_cast<u32x2*>(&dots[lane & 3][64 * chunk + 4 * (lane >> 2)]) =
        u32x2{pack2(dot[0], dot[1]), pack2(dot[2], dot[3])};
  }
  __syncthreads();
  const int qb = qb0 + wave;
  if (wave >= 4 || qb >= p.nq) return;
  const RowGeom g(p, qb, a.mg_hw, a.mg_nw);
  uint16_t* srow = a.scores ? a.scores + ((int64_t)bh * p.nq + qb) * nk : nullptr;
  uint32_t kr[KS];
  int nf = 0;
#pragma unroll
  for (int r = 0; r < KS; ++r) {
    const int j = r * 64 + lane;
    bool f = false;
    kr[r] = 0u;
    if (j < nk) kr[r] = finish_key<E>(p, g, srow, j, dots[wave][j], f, a.mg_hw, a.mg_nw);
    nf += wave_count(f);
  }
  select_row<KS>(a, [&](int r) LI_MASK_INLINE { return kr[r]; }, KS, nf, qb, bh, lane);
}

// Sets *flag when any of the n ids lies outside [0, n_blocks).  One read of the
// list, 16 ids per thread and pass; the flag (host memory) is written only when
// an id is out of range.
__global__ __launch_bounds__(256) void check_ids_kernel(const int32_t* ids, int64_t n, int32_t n_blocks, int32_t* flag) {
  typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
  const uint32_t lim = (uint32_t)n_blocks;
  const int64_t threads = (int64_t)gridDim.x * 256, me = (int64_t)blockIdx.x * 256 + threadIdx.x;
  bool bad = false;
  const int64_t n4 = n >> 2;  // the list starts 16-byte aligned
  int64_t i = me;
  for (; i + 3 * threads < n4; i += 4 * threads) {
    i32x4 x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = reinterpret_cast<const i32x4*>(ids)[i + k * threads];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= (uint32_t)x[k][e] >= lim;
  }
  for (; i < n4; i += threads) {
    const i32x4 x = reinterpret_cast<const i32x4*>(ids)[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) bad |= (uint32_t)x[e] >= lim;
  }
  if (me < (n & 3)) bad |= (uint32_t)ids[4 * n4 + me] >= lim;
  if (bad) __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr int kTiledMaxNk = 64 * 28;

}  // namespace
}  // namespace li

using namespace li;

extern "C" int li_block_mask(int dtype, int32_t B, int32_t NH, int32_t D, const void* q_pool,
                             const int64_t q_pool_strides[4], const void* k_pool, const int64_t k_pool_strides[4],
                             const li_mask_params* params, int32_t* indices, int32_t* counts, void* scores,
                             void* stream) {
  if (!q_pool || !k_pool || !q_pool_strides || !k_pool_strides || !params || !indices || !counts)
    return LI_ERR_INVALID_ARG;
  if (B <= 0 || NH <= 0) return LI_ERR_INVALID_ARG;
  const li_mask_params& p = *params;
  if (p.nq < 0 || p.nk < 0 || p.nh <= 0 || p.nw <= 0 || p.num_txt_blk < 0 || p.kmax < 0 || p.n_recent < 0)
    return LI_ERR_SHAPE;
  if (p.metric < LI_METRIC_COSINE || p.metric > LI_METRIC_DOT) return LI_ERR_INVALID_ARG;
  if (p.budget_mode != LI_BUDGET_HISTORY && p.budget_mode != LI_BUDGET_TOTAL) return LI_ERR_INVALID_ARG;
  if (!(p.topk_ratio >= 0.0) || p.topk_ratio > 1e6) return LI_ERR_INVALID_ARG;
  if (p.nk > kMaxNk) return LI_ERR_TOO_LARGE;
  if (p.kmax < p.num_txt_blk) return LI_ERR_SHAPE;
  if (p.nq == 0) return LI_OK;
  if ((int64_t)B * NH > 65535) return LI_ERR_SHAPE;
  MaskArgs a = {};
  a.qp = static_cast<const uint16_t*>(q_pool);
  a.kp = static_cast<const uint16_t*>(k_pool);
  for (int i = 0; i < 4; ++i) {
    a.qs[i] = q_pool_strides[i];
    a.ks[i] = k_pool_strides[i];
  }
  a.p = p;
  a.indices = indices;
  a.counts = counts;
  a.scores = static_cast<uint16_t*>(scores);
  a.NH = NH;
  const bool vec_k = k_pool_strides[3] == 1 && (reinterpret_cast<uintptr_t>(k_pool) & 15u) == 0 &&
                     k_pool_strides[0] % 8 == 0 && k_pool_strides[1] % 8 == 0 && k_pool_strides[2] % 8 == 0;
  // The shared-pool kernel keeps a chunk's row offsets in 32 bits.
  const bool shared = vec_k && p.nk > 0 && p.nk <= kTiledMaxNk && k_pool_strides[2] >= 0 &&
                      k_pool_strides[2] < (1ll << 24);
  const int64_t hw = (int64_t)p.nh * p.nw;
  a.mg_hw = hw < 65536 ? magic16((int32_t)hw) : 0x10000u;  // j / hw = 0 for every block
  a.mg_nw = p.nw < 65536 ? magic16(p.nw) : 0x10000u;
  // Generic path: per-wave LDS slice of nk keys + the query row, up to 4
  // waves (rows) per workgroup.
  const size_t per_wave = ((size_t)p.nk + D) * 4;
  int waves = (int)(65536 / per_wave);
  waves = waves < 1 ? 1 : (waves > 4 ? 4 : waves);
  const int rows = shared ? 4 : waves;
  const size_t lds = shared ? 0 : per_wave * waves;
  a.NBH = B * NH;
  a.groups = (p.nq + rows - 1) / rows;
  if (shared && (int64_t)a.groups * a.NBH > 0x7FFFFFFF) return LI_ERR_SHAPE;
  dim3 grid((unsigned)a.groups, (unsigned)(B * NH));
  if (shared) grid = dim3((unsigned)(a.groups * a.NBH));
  hipStream_t s = static_cast<hipStream_t>(stream);
  clear_launch_error();
  // Past 256 blocks eight scoring waves end a workgroup soonest, but hold a CU's
  // LDS (D = 128); once the row groups outnumber the CUs, four of them and two
  // workgroups a CU are faster.  Kernel times, us, SW = 8 and 4 (heads x rows x
  // blocks, scaled dot product):
  //   16 x 56 x 896 (224 groups)  18.7, 20.3     16 x 72 x 300 (288)   23.5, 16.2
  //    1 x 1000 x 1000 (250)      19.3, 20.8     16 x 156 x 600 (624)  44.0, 32.0
  //   16 x 64 x 300 (256)         14.1, 14.9     16 x 1000 x 512       194.2, 113.6
  // and D = 64, 8 x 300 x 300: 21.0, 17.3.  Past 1024 blocks SW = 4 does not fit twice
  // either (16 x 300 x 1500: 128.7, 141.0).
  const bool many = (int64_t)a.groups * a.NBH > device_cus();
#define LI_MASK_LAUNCH(E_, D_)                                                                           \
  do {                                                                                                   \
    if (shared && p.nk <= 256)                                                                           \
      hipLaunchKernelGGL((block_mask_rows_kernel<E_, D_, 4, 4>), grid, dim3(512), lds, s, a);            \
    else if (shared && p.nk <= 1024 && many)                                                             \
      hipLaunchKernelGGL((block_mask_rows_kernel<E_, D_, 16, 4>), grid, dim3(512), lds, s, a);           \
    else if (shared && p.nk <= 1024)                                                                     \
      hipLaunchKernelGGL((block_mask_rows_kernel<E_, D_, 16, 8>), grid, dim3(512), lds, s, a);           \
    else if (shared)                                                                                     \
      hipLaunchKernelGGL((block_mask_rows_kernel<E_, D_, 28, 8>), grid, dim3(512), lds, s, a);           \
    else                                                                                                 \
      hipLaunchKernelGGL((block_mask_kernel<E_, D_>), grid, dim3((unsigned)(64 * waves)), lds, s, a, waves); \
  } while (0)
  if (dtype == LI_DTYPE_BF16 && D == 128)
    LI_MASK_LAUNCH(Bf16, 128);
  else if (dtype == LI_DTYPE_BF16 && D == 64)
    LI_MASK_LAUNCH(Bf16, 64);
  else if (dtype == LI_DTYPE_F16 && D == 128)
    LI_MASK_LAUNCH(F16, 128);
  else if (dtype == LI_DTYPE_F16 && D == 64)
    LI_MASK_LAUNCH(F16, 64);
  else
    return LI_ERR_UNSUPPORTED;
#undef LI_MASK_LAUNCH
  return launch_status();
}

extern "C" int li_check_block_ids(const int32_t* ids, int64_t n, int32_t n_blocks, int32_t* flag, void* stream) {
  if (!ids || !flag || n < 0 || n_blocks < 0) return LI_ERR_INVALID_ARG;
  if ((reinterpret_cast<uintptr_t>(ids) & 15u) != 0) return LI_ERR_INVALID_ARG;
  if (n == 0) return LI_OK;
  const int64_t wgs = (n + 4095) / 4096;
  clear_launch_error();
  hipLaunchKernelGGL(check_ids_kernel, dim3((unsigned)(wgs < 512 ? wgs : 512)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), ids, n, n_blocks, flag);
  return launch_status();
}
