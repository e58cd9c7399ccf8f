// 3D (t,h,w) tile gather with fixed-order fp32 mean pooling, and its inverse
// scatter, for gfx950.
//
// Replaces the Triton kernels _fused_q_prep_kernel, _fused_kv_prep_kernel and
// _fused_untile_kernel (hy-worldplay/.../ar_sparse_operation.py:26-161; copies in
// bi_sparse_operation_for_KV_cache.py:27-163 and matrix-game-3.0/.../bi_sparse_operation.py:25-140).
//
// Index maps (ar_sparse_operation.py:42-59): block blk -> (ct, ch, cw) =
// (blk / (nh*nw), (blk / nw) % nh, blk % nw); tile row f -> (ft, fh, fw) =
// (f / (tw*th), (f / tw) % th, f % tw); token l = t*H*W + h*W + w.
//
// One launch takes up to kMaxJobs jobs, each a gather of one tensor into tiles
// (16-bit, or OCP e4m3 codes with one scale per tile block), its mean pool, or
// both: what an attention call needs of its queries, keys, values and text.
// One 256-thread workgroup per (tile, batch*head) of a job.  Thread t owns the
// 16-byte column chunk c = t % (D/8) (8 elements) of tile rows f = g, g+NG, ...
// with g = t / (D/8) and NG = 256 / (D/8): sixteen consecutive threads move one
// 256-byte token row, so every global access is a coalesced 16-byte vector
// access whenever the row is contiguous.  The pool sums each group's rows
// sequentially in fp32 from +0.0, then combines the NG partials with the
// pairwise tree s[g] += s[g + stride], stride = NG/2 .. 1, and divides by BS.
// That order is fixed so the pooled values are reproducible bit for bit.
#include "li_common.hpp"

namespace li {
namespace {

// Fields in the order of their use: a workgroup reads its job with scalar loads.
struct PrepJob {
  const uint16_t* src;
  int64_t ss[4];
  li_tile_geom g;
  uint32_t mg_tw, mg_th, mg_nw, mg_nh;  // udiv16 magics
  int32_t bs;
  int32_t vec_src, vec_dst, reserved;
  // Tiles at block blk + dst_off (null: none): 16-bit elements, or e4m3 codes
  // (byte strides) when `scale` is given, one fp32 scale per block.
  uint16_t* dst;
  float* scale;
  int64_t dst_off;
  int64_t ds[5];
  // Mean pool at block blk + pool_off (null: none) and, optionally, a second
  // copy with the same strides: each pooled row divided by its L2 norm as the
  // cosine block-mask metric normalises it.
  uint16_t* mean;
  uint16_t* mean_n;
  int64_t pool_off;
  int64_t ms[4];
  int64_t scs[3];
};

constexpr int kMaxJobs = 5;

struct PrepArgs {
  int32_t end[kMaxJobs];  // tile blocks of each job and the earlier ones
  int32_t NH;
  uint32_t mg_NH;
  int32_t rows;           // blocks along y
  PrepJob job[kMaxJobs];
};

__device__ __forceinline__ u32x4 load8(const uint16_t* p, int64_t stride, bool vec) {
  if (vec) return *reinterpret_cast<const u32x4*>(p);
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = pack2(p[(2 * i) * stride], p[(2 * i + 1) * stride]);
  return r;
}

__device__ __forceinline__ void store8(uint16_t* p, int64_t stride, bool vec, u32x4 v) {
  if (vec) {
    *reinterpret_cast<u32x4*>(p) = v;
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    p[(2 * i) * stride] = uint16_t(v[i] & 0xFFFFu);
    p[(2 * i + 1) * stride] = uint16_t(v[i] >> 16);
  }
}

// Workgroup -> (tile block, b*h) for a (blocks, B*NH) grid, heads fastest in
// dispatch order: the workgroups in flight together read the same tokens of
// every head, which with (B, L, H, D) token views is one contiguous span per
// token instead of one head's 2*D bytes of it.
__device__ __forceinline__ void tile_unit(int& blk, int& bh) {
  const uint64_t nbh = gridDim.y;
  const uint64_t lin = blockIdx.x + (uint64_t)gridDim.x * blockIdx.y;
  blk = (int)(lin / nbh);
  bh = (int)(lin - (uint64_t)blk * nbh);
}

// One block of a job.  VEC: every row of the source and the 16-bit tiles is
// moved with 16-byte vector accesses (unit innermost stride, 16-byte aligned
// rows).  The element-wise path for other strides is a separate instantiation,
// so the vector one does not carry its per-element address registers.
//
// e4m3 codes: amax = max |x| over the block (padding rows are zeros), scale =
// amax / 448, codes e4m3(x * (448 / amax)), both quotients correctly rounded in
// fp32; scale 1 and zero codes for an all-zero block.  After scaling no finite
// element exceeds 448 (1 + 2^-23), which rounds to 448, so v_cvt_pk_fp8_f32
// (round to nearest even) never saturates or yields NaN.  The whole block is
// held in registers for it (BS <= R NG rows, checked on the host): loads, then
// the workgroup's amax, then the stores.  The pool is always of the 16-bit
// values.
//
// `Job` is PrepJob in the constant address space: the job of a workgroup is
// indexed in the kernel-argument segment itself, whose fields are then scalar
// loads (indexing the by-value parameter would copy it to scratch).
//
// A pool is bound by the read of its tensor and by how soon a workgroup's loads
// go out, since a workgroup lives for one block: the grid has no division to
// undo (heads along x), block coordinates take udiv16, all row loads of a batch
// are unconditional (rows outside the grid read the block's first token, which
// is always inside, and are replaced by zeros), a row's offset from the block's
// first token takes 32 bits, and the job is read in one scalar round trip.  Both
// pools of the 16-head 30 x 52 call with 4 + 12 frames (103 MB): 21.2 us, against
// 21.8 with a kernel of its own for the pair and 24.1 with this one before those
// changes; the e4m3 tiles and pools of the same call with 200 text tokens (156
// MB): 31.8 us, against 43.2 in three launches and 19 in four more for padding
// the text.
typedef __attribute__((address_space(4))) const PrepJob Job;

template <typename E, int D, bool VEC>
__device__ __forceinline__ void prep_block(Job& a, int b, int h, int blk) {
  constexpr int CPR = D / 8;
  constexpr int NG = 256 / CPR;
  __shared__ float red[NG][D];
  __shared__ uint32_t wmax[4];

  const int tid = threadIdx.x;
  const int c = tid % CPR, g0 = tid / CPR;
  const int T = a.g.T, H = a.g.H, W = a.g.W, tt = a.g.tt, nh = a.g.nh, nw = a.g.nw, bs = a.bs;
  const uint32_t tw = a.g.tw, th = a.g.th, mg_tw = a.mg_tw, mg_th = a.mg_th, mg_nw = a.mg_nw, mg_nh = a.mg_nh;
  const uint16_t* src = a.src;
  const int64_t st_b = a.ss[0], st_h = a.ss[1], st_l = a.ss[2], st_d = VEC ? 1 : a.ss[3];
  uint16_t* dst = a.dst;
  float* scale = a.scale;
  uint16_t* mean = a.mean;
  // All of these are needed at once: without the empty asm the compiler reads
  // them where each is first used, one scalar round trip after the other.
  asm volatile("" ::"s"(T), "s"(H), "s"(W), "s"(tt), "s"(th), "s"(tw), "s"(nh), "s"(nw), "s"(bs), "s"(mg_tw), "s"(mg_th),
               "s"(mg_nw), "s"(mg_nh), "s"(src), "s"(st_b), "s"(st_h), "s"(st_l), "s"(dst), "s"(scale), "s"(mean));
  // VEC: fewer than 2^16 blocks (checked on the host).
  const uint32_t rem = VEC ? udiv16(blk, mg_nw) : (uint32_t)blk / (uint32_t)nw, cw = blk - rem * nw;
  const uint32_t ct = VEC ? udiv16(rem, mg_nh) : rem / (uint32_t)nh, ch = rem - ct * nh;
  const int t0 = ct * tt, h0 = ch * th, w0 = cw * tw;
  // Rows of the block inside the grid: ft < nt, fh < nhh, fw < nww.
  const uint32_t nt = T - t0, nhh = H - h0, nww = W - w0;
  const uint16_t* sbase = src + b * st_b + h * st_h + (((int64_t)t0 * H + h0) * W + w0) * st_l;
  const bool vs = VEC || a.vec_src != 0;

  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.0f;

  // R rows per thread in flight: all loads of a batch are issued before its
  // rows are stored and summed (in row order, so the sums do not depend on R).
  // VEC: one batch (checked on the host).
  constexpr int R = 8;
  int f0 = 0;
  do {
    u32x4 v[R];
    bool ok[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if constexpr (!VEC) {
        ok[i] = false;
        v[i] = u32x4{0u, 0u, 0u, 0u};
        if (f0 + i * NG >= bs) continue;  // the whole workgroup
      }
      const uint32_t f = f0 + i * NG + g0;
      const uint32_t r = udiv16(f, mg_tw), fw = f - r * tw;
      const uint32_t ft = udiv16(r, mg_th), fh = r - ft * th;
      ok[i] = (f < (uint32_t)bs) & (ft < nt) & (fh < nhh) & (fw < nww);
      const uint32_t l = ok[i] ? (ft * H + fh) * W + fw : 0u;
      // VEC: a row's byte offset from the block's first token is below 2^31
      // (checked on the host).
      if constexpr (VEC)
        v[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(sbase) + (l * (uint32_t)(2 * st_l) + 16u * c));
      else {
        // A row at a time, and only rows that are there: with the element loads of
        // eight rows in flight at once the kernel takes 226 VGPRs, and rows outside
        // the block (three in four of a 64-row block at D = 64) would cost as much
        // as the others: tiles and pool of 16 heads x 12 frames x 30 x 52 97.1 us
        // that way, 78.2 this way; K and V of 8 heads x 2 x 32 x 32 at D = 64 23.2, 8.3.
        if (ok[i]) v[i] = load8(sbase + (int64_t)l * st_l + (int64_t)(8 * c) * st_d, st_d, vs);
        asm volatile("" : "+v"(v[i])::"memory");
      }
    }
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (!ok[i]) v[i] = u32x4{0u, 0u, 0u, 0u};
    }
    if (dst) {
      const int64_t doff = b * a.ds[0] + h * a.ds[1] + (blk + a.dst_off) * a.ds[2];
      if (scale) {
        // Largest magnitude: for finite 16-bit floats the magnitude bits order
        // as the values do.
        uint32_t mb = 0;
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t x = v[i][e];
            mb = __builtin_elementwise_max(mb, __builtin_elementwise_max(x & 0x7FFFu, (x >> 16) & 0x7FFFu));
          }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) mb = __builtin_elementwise_max(mb, (uint32_t)__shfl_xor((int)mb, o));
        if ((tid & 63) == 0) wmax[tid >> 6] = mb;
        __syncthreads();
        mb = __builtin_elementwise_max(__builtin_elementwise_max(wmax[0], wmax[1]),
                                       __builtin_elementwise_max(wmax[2], wmax[3]));
        const float amax = E::to_f32((uint16_t)mb);
        const bool zero = !(amax > 0.0f);
        const float inv = zero ? 1.0f : 448.0f / amax;
        if (tid == 0)
          scale[b * a.scs[0] + h * a.scs[1] + (blk + a.dst_off) * a.scs[2]] = zero ? 1.0f : amax / 448.0f;
        uint8_t* dbase = reinterpret_cast<uint8_t*>(dst) + doff + 8 * c;
#pragma unroll
        for (int i = 0; i < R; ++i) {
          const int f = f0 + i * NG + g0;
          u32x2 q;
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            const uint32_t lo = v[i][2 * p], hi = v[i][2 * p + 1];
            int w = __builtin_amdgcn_cvt_pk_fp8_f32(E::to_f32(uint16_t(lo & 0xFFFFu)) * inv,
                                                    E::to_f32(uint16_t(lo >> 16)) * inv, 0, false);
            w = __builtin_amdgcn_cvt_pk_fp8_f32(E::to_f32(uint16_t(hi & 0xFFFFu)) * inv,
                                                E::to_f32(uint16_t(hi >> 16)) * inv, w, true);
            q[p] = (uint32_t)w;
          }
          if (f < bs) *reinterpret_cast<u32x2*>(dbase + (int64_t)f * a.ds[3]) = q;
        }
      } else {
        const int64_t dt_d = VEC ? 1 : a.ds[4];
        const bool vd = VEC || a.vec_dst != 0;
        uint16_t* dbase = dst + doff + (int64_t)(8 * c) * dt_d;
#pragma unroll
        for (int i = 0; i < R; ++i) {
          const int f = f0 + i * NG + g0;
          if (f < bs) store8(dbase + (int64_t)f * a.ds[3], dt_d, vd, v[i]);
        }
      }
    }
    if (mean) {
      // Rows past the block's end are zeros: adding them changes nothing.
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[2 * e] = acc[2 * e] + E::to_f32(uint16_t(v[i][e] & 0xFFFFu));
          acc[2 * e + 1] = acc[2 * e + 1] + E::to_f32(uint16_t(v[i][e] >> 16));
        }
    }
    f0 += R * NG;
  } while (!VEC && f0 < bs);
  if (!mean) return;

#pragma unroll
  for (int i = 0; i < 8; ++i) red[g0][8 * c + i] = acc[i];
  __syncthreads();
  const int64_t moff = b * a.ms[0] + h * a.ms[1] + (blk + a.pool_off) * a.ms[2], mt_d = a.ms[3];
  float mrow = 0.0f;
  if (tid < D) {
    float s[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) s[i] = red[i][tid];
#pragma unroll
    for (int stride = NG / 2; stride >= 1; stride /= 2) {
#pragma unroll
      for (int i = 0; i < stride; ++i) s[i] = s[i] + s[i + stride];
    }
    const uint16_t m = E::from_f32(s[0] / (float)bs);
    mean[moff + (int64_t)tid * mt_d] = m;
    mrow = E::to_f32(m);
  }
  if (a.mean_n) {
    // The cosine metric's normalisation of the rounded row: sequential fp32
    // sum of squares over d from +0.0, x / max(E(sqrt(.)), E(1e-12)), the
    // arithmetic the block mask applies to a raw key pool row.
    __syncthreads();  // the partial sums are read
    if (tid < D) red[0][tid] = mrow;
    __syncthreads();
    // Wave 0 alone finishes the row (every lane runs the same chain over
    // broadcast reads); the other waves end here and free their slots.
    if (tid >= 64) return;
    float ss = 0.0f;
#pragma unroll
    for (int d = 0; d < D; ++d) ss = ss + red[0][d] * red[0][d];
    const float nrm = E::to_f32(E::from_f32(__builtin_sqrtf(ss)));
    const float eps = E::to_f32(E::from_f32(1e-12f));
    const float den = nrm > eps ? nrm : eps;
#pragma unroll
    for (int d = tid; d < D; d += 64) a.mean_n[moff + (int64_t)d * mt_d] = E::from_f32(red[0][d] / den);
  }
}

// The jobs' tile blocks follow each other along y (and z, past 32768 blocks);
// x = b * NH + h runs fastest, so the workgroups in flight together read the
// same tokens of every head, which with (B, L, H, D) token views is one
// contiguous span per token instead of one head's 2*D bytes of it.
template <typename E, int D, bool VEC>
__global__ __launch_bounds__(256, VEC ? 8 : 2) void prep_kernel(PrepArgs) {
  typedef __attribute__((address_space(4))) const PrepArgs Args;
  Args& a = *(Args*)__builtin_amdgcn_kernarg_segment_ptr();
  const int e0 = a.end[0], e1 = a.end[1], e2 = a.end[2], e3 = a.end[3], total = a.end[4], NH = a.NH, rows = a.rows;
  const uint32_t mg_NH = a.mg_NH;
  asm volatile("" ::"s"(e0), "s"(e1), "s"(e2), "s"(e3), "s"(total), "s"(NH), "s"(rows), "s"(mg_NH));  // one read
  const int bh = blockIdx.x, blk = blockIdx.z * rows + blockIdx.y;
  if (blk >= total) return;
  const int j = (blk >= e0) + (blk >= e1) + (blk >= e2) + (blk >= e3);
  const int first = blk >= e3 ? e3 : blk >= e2 ? e2 : blk >= e1 ? e1 : blk >= e0 ? e0 : 0;
  const int b = (int)udiv16(bh, mg_NH), h = bh - b * NH;
  prep_block<E, D, VEC>(a.job[j], b, h, blk - first);
}

struct UntileArgs {
  const uint16_t* src;
  int64_t ss[5];
  uint16_t* dst;
  int64_t ds[4];
  int32_t NH, bs;
  li_tile_geom g;
  int32_t vec_src, vec_dst;
};

template <int D, bool VEC>
__global__ __launch_bounds__(256) void untile_kernel(UntileArgs a) {
  constexpr int CPR = D / 8;
  constexpr int NG = 256 / CPR;
  int blk, bh;
  tile_unit(blk, bh);
  const int b = bh / a.NH, h = bh % a.NH;
  const int tid = threadIdx.x;
  const int c = tid % CPR, g0 = tid / CPR;
  const li_tile_geom& g = a.g;
  const int cw = blk % g.nw, rem = blk / g.nw;
  const int ch = rem % g.nh, ct = rem / g.nh;
  const bool vs = VEC || a.vec_src != 0, vd = VEC || a.vec_dst != 0;
  const uint16_t* sbase = a.src + b * a.ss[0] + h * a.ss[1] + blk * a.ss[2] + (int64_t)(8 * c) * a.ss[4];
  uint16_t* dbase = a.dst + b * a.ds[0] + h * a.ds[1] + (int64_t)(8 * c) * a.ds[3];
  for (int f = g0; f < a.bs; f += NG) {
    const int fw = f % g.tw, r = f / g.tw;
    const int fh = r % g.th, ft = r / g.th;
    const int t = ct * g.tt + ft, hh = ch * g.th + fh, w = cw * g.tw + fw;
    if ((t < g.T) && (hh < g.H) && (w < g.W)) {
      const int64_t l = (int64_t)t * g.H * g.W + (int64_t)hh * g.W + w;
      u32x4 v = load8(sbase + (int64_t)f * a.ss[3], a.ss[4], vs);
      store8(dbase + l * a.ds[2], a.ds[3], vd, v);
    }
  }
}

// 16-byte vector access is legal when the innermost stride is 1 and every row
// start (and the base pointer) is 16-byte aligned.
bool vec_ok(const void* p, const int64_t* strides, int nd) {
  if (strides[nd - 1] != 1) return false;
  if ((reinterpret_cast<uintptr_t>(p) & 15u) != 0) return false;
  for (int i = 0; i < nd - 1; ++i)
    if (strides[i] % 8 != 0) return false;
  return true;
}

int check_geom(const li_tile_geom* g) {
  if (!g) return LI_ERR_INVALID_ARG;
  if (g->T < 0 || g->H <= 0 || g->W <= 0 || g->tt <= 0 || g->th <= 0 || g->tw <= 0) return LI_ERR_SHAPE;
  if (g->nh != (g->H + g->th - 1) / g->th || g->nw != (g->W + g->tw - 1) / g->tw) return LI_ERR_SHAPE;
  return LI_OK;
}

int64_t num_blocks(const li_tile_geom* g) { return (int64_t)((g->T + g->tt - 1) / g->tt) * g->nh * g->nw; }

bool prep_supported(int dtype, int32_t D) {
  return (dtype == LI_DTYPE_BF16 || dtype == LI_DTYPE_F16) && (D == 128 || D == 64);
}

// Runs up to kMaxJobs jobs (their src, dst, scale and mean fields set) over the
// geometries `geoms`: in one launch, or two when only some of them can be moved
// with vector accesses.  Jobs without tile blocks are dropped.
int launch_prep(int dtype, int32_t B, int32_t NH, int32_t D, const PrepArgs& jobs, const li_tile_geom* const* geoms,
                int n, hipStream_t stream) {
  if (B <= 0 || NH <= 0) return LI_ERR_INVALID_ARG;
  PrepArgs a[2] = {};  // element-wise, vector
  int64_t total[2] = {0, 0};
  int live[2] = {0, 0};
  for (int i = 0; i < n; ++i) {
    const li_tile_geom* geom = geoms[i];
    const int st = check_geom(geom);
    if (st != LI_OK) return st;
    const int64_t blocks = num_blocks(geom);
    if (blocks == 0) continue;
    if (blocks > 0x7FFFFFFF || (int64_t)B * NH > 65535) return LI_ERR_SHAPE;
    if ((int64_t)geom->tt * geom->th * geom->tw >= 65536) return LI_ERR_SHAPE;
    PrepJob job = jobs.job[i];
    job.g = *geom;
    job.bs = geom->tt * geom->th * geom->tw;
    job.mg_tw = magic16(geom->tw);
    job.mg_th = magic16(geom->th);
    job.mg_nw = magic16(geom->nw);
    job.mg_nh = magic16(geom->nh);
    job.vec_src = vec_ok(job.src, job.ss, 4);
    job.vec_dst = !job.dst || job.scale ? 1 : vec_ok(job.dst, job.ds, 5);
    if (!prep_supported(dtype, D)) return LI_ERR_UNSUPPORTED;
    // An e4m3 block is held in registers: at most 8 rows per thread.
    if (job.scale && job.bs > 8 * (256 / (D / 8))) return LI_ERR_UNSUPPORTED;
    // The vector kernel takes a block in one batch of 8 rows per thread, holds a
    // row's byte offset from its block's first token in 32 bits, and block
    // numbers in 16.
    const int64_t rows = (int64_t)(geom->tt - 1) * geom->H * geom->W + (int64_t)(geom->th - 1) * geom->W + geom->tw;
    const bool near = job.ss[2] >= 0 && job.ss[2] < (1ll << 30) && rows < (1ll << 30) && rows * job.ss[2] < (1ll << 29);
    const int v = job.vec_src && job.vec_dst && near && blocks < 65536 &&
                          job.bs <= 8 * (256 / (D / 8)) ? 1 : 0;
    total[v] += blocks;
    if (total[v] > 0x7FFFFFFF) return LI_ERR_SHAPE;
    a[v].end[live[v]] = (int32_t)total[v];
    a[v].job[live[v]++] = job;
  }
  for (int v = 0; v < 2; ++v) {
    if (live[v] == 0) continue;
    for (int i = live[v]; i < kMaxJobs; ++i) a[v].end[i] = (int32_t)total[v];
    a[v].NH = NH;
    a[v].mg_NH = magic16(NH);
    const unsigned rows = (unsigned)(total[v] < 32768 ? total[v] : 32768);
    a[v].rows = (int32_t)rows;
    const dim3 grid((unsigned)(B * NH), rows, (unsigned)((total[v] + rows - 1) / rows));
    clear_launch_error();
#define LI_PREP_LAUNCH(E_, D_)                                                                \
  do {                                                                                        \
    if (v)                                                                                    \
      hipLaunchKernelGGL((prep_kernel<E_, D_, true>), grid, dim3(256), 0, stream, a[v]);      \
    else                                                                                      \
      hipLaunchKernelGGL((prep_kernel<E_, D_, false>), grid, dim3(256), 0, stream, a[v]);     \
  } while (0)
    if (dtype == LI_DTYPE_BF16 && D == 128)
      LI_PREP_LAUNCH(Bf16, 128);
    else if (dtype == LI_DTYPE_BF16)
      LI_PREP_LAUNCH(Bf16, 64);
    else if (D == 128)
      LI_PREP_LAUNCH(F16, 128);
    else
      LI_PREP_LAUNCH(F16, 64);
#undef LI_PREP_LAUNCH
    const int st = launch_status();
    if (st != LI_OK) return st;
  }
  return LI_OK;
}

template <size_t N>
void copy_strides(int64_t (&to)[N], const int64_t* from) {
  for (size_t i = 0; i < N; ++i) to[i] = from[i];
}

void set_src(PrepJob& j, const void* src, const int64_t* ss) {
  j.src = static_cast<const uint16_t*>(src);
  copy_strides(j.ss, ss);
}

void set_dst(PrepJob& j, void* dst, const int64_t* ds, int64_t dst_off) {
  j.dst = static_cast<uint16_t*>(dst);
  copy_strides(j.ds, ds);
  j.dst_off = dst_off;
}

void set_scale(PrepJob& j, float* scale, const int64_t* scs) {
  j.scale = scale;
  copy_strides(j.scs, scs);
}

void set_mean(PrepJob& j, void* mean, void* mean_n, const int64_t* ms, int64_t pool_off) {
  j.mean = static_cast<uint16_t*>(mean);
  j.mean_n = static_cast<uint16_t*>(mean_n);
  copy_strides(j.ms, ms);
  j.pool_off = pool_off;
}

// e4m3 tile rows: unit d stride, 8-byte aligned rows; one scale per block.
bool fp8_dst_ok(const void* p, const int64_t st[5]) {
  return p && (reinterpret_cast<uintptr_t>(p) & 7u) == 0 && st[4] == 1 && st[0] % 8 == 0 && st[1] % 8 == 0 &&
         st[2] % 8 == 0 && st[3] % 8 == 0;
}

}  // namespace
}  // namespace li

using namespace li;

extern "C" int li_q_prep(int dtype, int32_t B, int32_t NH, int32_t D, const void* src, const int64_t src_strides[4],
                         void* dst, const int64_t dst_strides[5], void* mean, const int64_t mean_strides[4],
                         const li_tile_geom* geom, void* stream) {
  if (!src || !dst || !mean || !src_strides || !dst_strides || !mean_strides) return LI_ERR_INVALID_ARG;
  PrepArgs a = {};
  set_src(a.job[0], src, src_strides);
  set_dst(a.job[0], dst, dst_strides, 0);
  set_mean(a.job[0], mean, nullptr, mean_strides, 0);
  return launch_prep(dtype, B, NH, D, a, &geom, 1, static_cast<hipStream_t>(stream));
}

extern "C" int li_kv_prep(int dtype, int32_t B, int32_t NH, int32_t D, const void* k_src,
                          const int64_t k_src_strides[4], const void* v_src, const int64_t v_src_strides[4],
                          void* k_dst, const int64_t k_dst_strides[5], void* v_dst, const int64_t v_dst_strides[5],
                          void* k_mean, const int64_t mean_strides[4], int64_t dst_off, int64_t pool_off,
                          const li_tile_geom* geom, void* stream) {
  if (!k_src || !v_src || !k_dst || !v_dst || !k_mean || !k_src_strides || !v_src_strides || !k_dst_strides ||
      !v_dst_strides || !mean_strides)
    return LI_ERR_INVALID_ARG;
  if (dst_off < 0 || pool_off < 0) return LI_ERR_INVALID_ARG;
  PrepArgs a = {};
  set_src(a.job[0], k_src, k_src_strides);
  set_dst(a.job[0], k_dst, k_dst_strides, dst_off);
  set_mean(a.job[0], k_mean, nullptr, mean_strides, pool_off);
  set_src(a.job[1], v_src, v_src_strides);
  set_dst(a.job[1], v_dst, v_dst_strides, dst_off);
  const li_tile_geom* geoms[2] = {geom, geom};
  return launch_prep(dtype, B, NH, D, a, geoms, 2, static_cast<hipStream_t>(stream));
}

extern "C" int li_pool(int dtype, int32_t B, int32_t NH, int32_t D, const void* src, const int64_t src_strides[4],
                       void* mean, const int64_t mean_strides[4], int64_t pool_off, const li_tile_geom* geom,
                       void* stream) {
  if (!src || !mean || !src_strides || !mean_strides) return LI_ERR_INVALID_ARG;
  if (pool_off < 0) return LI_ERR_INVALID_ARG;
  PrepArgs a = {};
  set_src(a.job[0], src, src_strides);
  set_mean(a.job[0], mean, nullptr, mean_strides, pool_off);
  return launch_prep(dtype, B, NH, D, a, &geom, 1, static_cast<hipStream_t>(stream));
}

extern "C" int li_prep(int dtype, int32_t B, int32_t NH, int32_t D, const li_prep_job* jobs, int32_t n_jobs,
                       void* stream) {
  if (!jobs || n_jobs < 1 || n_jobs > kMaxJobs) return LI_ERR_INVALID_ARG;
  PrepArgs a = {};
  const li_tile_geom* geoms[kMaxJobs];
  for (int i = 0; i < n_jobs; ++i) {
    const li_prep_job& j = jobs[i];
    if (!j.src || (!j.dst && !j.mean) || (j.scales && !j.dst) || (j.mean_normalized && !j.mean) || j.dst_off < 0 ||
        j.pool_off < 0)
      return LI_ERR_INVALID_ARG;
    if (j.scales && !fp8_dst_ok(j.dst, j.dst_strides)) return LI_ERR_INVALID_ARG;
    set_src(a.job[i], j.src, j.src_strides);
    if (j.dst) set_dst(a.job[i], j.dst, j.dst_strides, j.dst_off);
    if (j.scales) set_scale(a.job[i], j.scales, j.scale_strides);
    if (j.mean) set_mean(a.job[i], j.mean, j.mean_normalized, j.mean_strides, j.pool_off);
    geoms[i] = &j.geom;
  }
  return launch_prep(dtype, B, NH, D, a, geoms, n_jobs, static_cast<hipStream_t>(stream));
}

extern "C" int li_untile(int dtype, int32_t B, int32_t NH, int32_t D, const void* src, const int64_t src_strides[5],
                         void* dst, const int64_t dst_strides[4], const li_tile_geom* geom, void* stream) {
  if (!src || !dst || !src_strides || !dst_strides) return LI_ERR_INVALID_ARG;
  if (B <= 0 || NH <= 0) return LI_ERR_INVALID_ARG;
  if (dtype != LI_DTYPE_BF16 && dtype != LI_DTYPE_F16) return LI_ERR_UNSUPPORTED;
  int st = check_geom(geom);
  if (st != LI_OK) return st;
  const int64_t nblk = num_blocks(geom);
  if (nblk == 0) return LI_OK;
  if (nblk > 0x7FFFFFFF || (int64_t)B * NH > 65535) return LI_ERR_SHAPE;
  UntileArgs a = {};
  a.src = static_cast<const uint16_t*>(src);
  a.dst = static_cast<uint16_t*>(dst);
  for (int i = 0; i < 5; ++i) a.ss[i] = src_strides[i];
  for (int i = 0; i < 4; ++i) a.ds[i] = dst_strides[i];
  a.NH = NH;
  a.bs = geom->tt * geom->th * geom->tw;
  a.g = *geom;
  a.vec_src = vec_ok(src, src_strides, 5);
  a.vec_dst = vec_ok(dst, dst_strides, 4);
  dim3 grid((unsigned)nblk, (unsigned)(B * NH));
  hipStream_t s = static_cast<hipStream_t>(stream);
  clear_launch_error();
  const bool vec = a.vec_src && a.vec_dst;
  if (D == 128 && vec)
    hipLaunchKernelGGL((untile_kernel<128, true>), grid, dim3(256), 0, s, a);
  else if (D == 128)
    hipLaunchKernelGGL((untile_kernel<128, false>), grid, dim3(256), 0, s, a);
  else if (D == 64 && vec)
    hipLaunchKernelGGL((untile_kernel<64, true>), grid, dim3(256), 0, s, a);
  else if (D == 64)
    hipLaunchKernelGGL((untile_kernel<64, false>), grid, dim3(256), 0, s, a);
  else
    return LI_ERR_UNSUPPORTED;
  return launch_status();
}

extern "C" int li_tile_prep_fp8(int dtype, int32_t B, int32_t NH, int32_t D, const void* src,
                                const int64_t src_strides[4], void* dst, const int64_t dst_strides[5],
                                float* scales, const int64_t scale_strides[3], void* mean,
                                const int64_t mean_strides[4], int64_t dst_off, int64_t pool_off,
                                const li_tile_geom* geom, void* stream) {
  if (!src || !src_strides || !dst_strides || !scales || !scale_strides || (mean && !mean_strides))
    return LI_ERR_INVALID_ARG;
  if (dst_off < 0 || pool_off < 0 || !fp8_dst_ok(dst, dst_strides)) return LI_ERR_INVALID_ARG;
  PrepArgs a = {};
  set_src(a.job[0], src, src_strides);
  set_dst(a.job[0], dst, dst_strides, dst_off);
  set_scale(a.job[0], scales, scale_strides);
  if (mean) set_mean(a.job[0], mean, nullptr, mean_strides, pool_off);
  return launch_prep(dtype, B, NH, D, a, &geom, 1, static_cast<hipStream_t>(stream));
}

extern "C" int li_kv_prep_fp8(int dtype, int32_t B, int32_t NH, int32_t D, const void* k_src,
                              const int64_t k_src_strides[4], const void* v_src, const int64_t v_src_strides[4],
                              void* k_dst, const int64_t k_dst_strides[5], float* k_scales,
                              const int64_t k_scale_strides[3], void* v_dst, const int64_t v_dst_strides[5],
                              void* k_mean, const int64_t mean_strides[4], int64_t dst_off, int64_t pool_off,
                              const li_tile_geom* geom, void* stream) {
  if (!k_src || !v_src || !v_dst || !k_mean || !k_src_strides || !v_src_strides || !k_dst_strides ||
      !v_dst_strides || !mean_strides || !k_scales || !k_scale_strides)
    return LI_ERR_INVALID_ARG;
  if (dst_off < 0 || pool_off < 0 || !fp8_dst_ok(k_dst, k_dst_strides)) return LI_ERR_INVALID_ARG;
  PrepArgs a = {};
  set_src(a.job[0], k_src, k_src_strides);
  set_dst(a.job[0], k_dst, k_dst_strides, dst_off);
  set_scale(a.job[0], k_scales, k_scale_strides);
  set_mean(a.job[0], k_mean, nullptr, mean_strides, pool_off);
  set_src(a.job[1], v_src, v_src_strides);
  set_dst(a.job[1], v_dst, v_dst_strides, dst_off);
  const li_tile_geom* geoms[2] = {geom, geom};
  return launch_prep(dtype, B, NH, D, a, geoms, 2, static_cast<hipStream_t>(stream));
}

extern "C" int li_pool_pair(int dtype, int32_t B, int32_t NH, int32_t D, const void* src0,
                            const int64_t src0_strides[4], void* mean0, const int64_t mean0_strides[4],
                            int64_t pool_off0, const li_tile_geom* geom0, const void* src1,
                            const int64_t src1_strides[4], void* mean1, const int64_t mean1_strides[4],
                            int64_t pool_off1, const li_tile_geom* geom1, void* mean1_normalized,
                            void* stream) {
  if (!src0 || !mean0 || !src0_strides || !mean0_strides || !src1 || !mean1 || !src1_strides || !mean1_strides ||
      pool_off0 < 0 || pool_off1 < 0 || B <= 0 || NH <= 0)
    return LI_ERR_INVALID_ARG;
  if (check_geom(geom0) != LI_OK) return check_geom(geom0);
  if (check_geom(geom1) != LI_OK) return check_geom(geom1);
  if (!prep_supported(dtype, D)) return LI_ERR_UNSUPPORTED;  // also with no blocks to pool
  PrepArgs a = {};
  set_src(a.job[0], src0, src0_strides);
  set_mean(a.job[0], mean0, nullptr, mean0_strides, pool_off0);
  set_src(a.job[1], src1, src1_strides);
  set_mean(a.job[1], mean1, mean1_normalized, mean1_strides, pool_off1);
  const li_tile_geom* geoms[2] = {geom0, geom1};
  return launch_prep(dtype, B, NH, D, a, geoms, 2, static_cast<hipStream_t>(stream));
}
