// dugma_energy.hip -- convolved-uncertainty energy, fused pose adjoint,
// per-point adjoint and the finite-difference ("plain") gradient.
//
// Kernel shape (k_near): a workgroup takes 64 stationary points, one per lane
// of each of its 8 waves (the transformed sources in the pose and energy passes;
// targets, then sources, in the two per-point passes), finds the points of the
// other cloud that any of them can have a term other than exactly 0 with, and
// sums those pairs.  Per-pair terms are FP32, summed in FP32 over sub-tiles of
// kSub streamed points in their own order and then in FP64 per lane;
// workgroup partials are reduced in a fixed order, so results are
// deterministic run to run.  Nothing of size N x M is stored.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "dugma_internal.h"
#include "dugma_near.h"
#include "dugma_pairs.h"

namespace dugma {

constexpr int kBlock = 256;  // 4 waves of 64
constexpr int kSub = 64;     // FP32 sub-tile length before the FP64 flush
constexpr int kMinChunk = 32;  // fewest streamed points per chunk

// kModeHess: the pose pass plus the sums of an approximate pose Hessian
// (3-D, transformed sources stationary)
enum { kModeEnergy = 0, kModePose = 1, kModePoint = 2, kModeHess = 3 };
constexpr int kHessPart = 32;  // doubles per workgroup of k_hess_tiles (21 used)

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Entry (i <= j) of the Hessian of E for moving a stationary point p by
// p - t -> p - t + theta x (p - t) + delta, from its sums a = [E, EW (3), B
// (6, upper triangle)] with d = p - q: with z = p - t and J = [-[z]x | I],
// H = J^T B J plus -1/2 (EW z^T + z EW^T) + (EW . z) I in the theta block
// (the second-order turn of z).  The turn of p's own covariance enters only
// the gradient.  FP32: the Hessian only shapes the search direction.
__device__ __forceinline__ float point_hessian_entry(int i, int j, const float *z, const float *a) {
  auto Bm = [&](int u, int v) -> float {
    const int lo = u < v ? u : v, hi = u < v ? v : u;
    return a[4 + (lo == 0 ? hi : lo == 1 ? 2 + hi : 5)];
  };
  auto Mm = [&](int u, int v) -> float {  // [z]x
    if (u == v) return 0.0f;
    const int w = 3 - u - v;
    return ((u + 1) % 3 == v) ? -z[w] : z[w];
  };
  if (i >= 3) return Bm(i - 3, j - 3);
  if (j >= 3) {
    const int c = j - 3;
    return Mm(i, 0) * Bm(0, c) + Mm(i, 1) * Bm(1, c) + Mm(i, 2) * Bm(2, c);
  }
  float v = 0.0f;
  for (int u = 0; u < 3; ++u)
    for (int w = 0; w < 3; ++w) v += Mm(u, i) * Bm(u, w) * Mm(w, j);
  const float ez = a[1] * z[0] + a[2] * z[1] + a[3] * z[2];
  return v - 0.5f * (a[1 + i] * z[j] + z[i] * a[1 + j]) + (i == j ? ez : 0.0f);
}

struct PoseArg {
  double R[9];  // column-major
  double t[3];
};

// ---------------------------------------------------------------------------
// Per-call source records: x' = R x + t and S' = R S R^T in FP64, then
// split to FP32 hi/lo (positions) and rounded (covariance).
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ void transform_pos(const double *__restrict__ s, const PoseArg &ps, float *hi, float *lo) {
#pragma unroll
  for (int a = 0; a < D; ++a) {
    double v = ps.t[a];
#pragma unroll
    for (int b = 0; b < D; ++b) v = fma(ps.R[a + D * b], s[b], v);
    hi[a] = (float)v;
    lo[a] = (float)(v - (double)hi[a]);
  }
}
// S' = R S R^T (column-major)
template <int D>
__device__ __forceinline__ void transform_cov(const double *__restrict__ S, const PoseArg &ps, double *Sp) {
  double RS[9];
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int c = 0; c < D; ++c) {
      double v = 0.0;
#pragma unroll
      for (int b = 0; b < D; ++b) v = fma(ps.R[a + D * b], S[b + D * c], v);
      RS[a + D * c] = v;
    }
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int c = 0; c < D; ++c) {
      double v = 0.0;
#pragma unroll
      for (int b = 0; b < D; ++b) v = fma(RS[a + D * b], ps.R[c + D * b], v);
      Sp[a + D * c] = v;
    }
}
__device__ __forceinline__ void transform_rec(const double *__restrict__ s, const PoseArg &ps, Rec3I &r) {
  float hi[3], lo[3];
  transform_pos<3>(s, ps, hi, lo);
  r.hx = hi[0]; r.hy = hi[1]; r.hz = hi[2];
  r.lx = lo[0]; r.ly = lo[1]; r.lz = lo[2];
  r.s = (float)(s[3] * kLn4);
  r.pad0 = 0.0f;
}
__device__ __forceinline__ void transform_rec(const double *__restrict__ s, const PoseArg &ps, Rec2I &r) {
  float hi[3], lo[3];
  transform_pos<2>(s, ps, hi, lo);
  r.hx = hi[0]; r.hy = hi[1]; r.lx = lo[0]; r.ly = lo[1];
  r.s = (float)(s[2] * kLn4);
  r.pad0 = r.pad1 = r.pad2 = 0.0f;
}
__device__ __forceinline__ void transform_rec(const double *__restrict__ s, const PoseArg &ps, Rec3F &r) {
  float hi[3], lo[3];
  double Sp[9];
  transform_pos<3>(s, ps, hi, lo);
  transform_cov<3>(s + 3, ps, Sp);
  r.hx = hi[0]; r.hy = hi[1]; r.hz = hi[2];
  r.lx = lo[0]; r.ly = lo[1]; r.lz = lo[2];
  r.s11 = (float)Sp[0];
  r.s22 = (float)Sp[4];
  r.s33 = (float)Sp[8];
  r.s12 = (float)(0.5 * (Sp[3] + Sp[1]));
  r.s13 = (float)(0.5 * (Sp[6] + Sp[2]));
  r.s23 = (float)(0.5 * (Sp[7] + Sp[5]));
  r.pad0 = r.pad1 = r.pad2 = r.pad3 = 0.0f;
}
__device__ __forceinline__ void transform_rec(const double *__restrict__ s, const PoseArg &ps, Rec2F &r) {
  float hi[3], lo[3];
  double Sp[9];
  transform_pos<2>(s, ps, hi, lo);
  transform_cov<2>(s + 2, ps, Sp);
  r.hx = hi[0]; r.hy = hi[1]; r.lx = lo[0]; r.ly = lo[1];
  r.s11 = (float)Sp[0];
  r.s22 = (float)Sp[3];
  r.s12 = (float)(0.5 * (Sp[2] + Sp[1]));
  r.pad0 = 0.0f;
}

template <class Rec>
__global__ __launch_bounds__(kBlock) void k_transform_src(
    const double *__restrict__ src, int n, PoseArg ps, Rec *__restrict__ out) {
  constexpr int D = RecTraits<Rec>::D;
  const int k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= n) return;
  Rec r;
  transform_rec(src + (size_t)k * (D + D * D), ps, r);
  out[k] = r;
}

// ---------------------------------------------------------------------------
// Pair kernel
// ---------------------------------------------------------------------------
// One workgroup (8 waves) takes 64 stationary points that are neighbours in
// Hilbert order, one per lane of every wave, and the part qc of qsplit of the
// streamed cloud's sub-tiles (groups of up to kSub consecutive points, the FP32
// sums' unit).
//
// 1. Wave 0 reads the stationary points (XSRC: transforms them from the FP64
//    source data, so that no launch has to do it first) and leaves them and
//    the boxes of their 4 rows of 16 and 16 quads of 4 in LDS.
// 2. The lanes test the streamed cloud's 64-point boxes against the rows, then
//    the points of the boxes that are near against rows and quads, and set a
//    bit in LDS for each point that any of the 64 lanes may have a term other
//    than 0 with.  Bits stand in the streamed points' own order, group by
//    group.
// 3. Each wave turns its groups' set bits into a list (LDS), takes 64 entries
//    at a time -- lane l puts the record of entry l into LDS, every lane then
//    reads them one by one (LdsRecs) -- and adds their pairs one after another.
//    Points without a bit add exactly 0 for every lane, so the FP32 sums of a
//    group are those of all its points, in their order.
//
// What bounds it: at 200K x 200K (isotropic, 8-NN sigma) a workgroup lists 3,250
// of 200,000 streamed points, 1,450 of which any one lane needs, in 2,000
// sub-tiles: VALU issue (407 M wave instructions at 4 cycles: 203 M of the
// pairs, 80 M of the FP64 flushes, 124 M of finding the points).  0.63 ms;
// 18.4 ms with every pair evaluated (outputs equal to 2e-16), 0.69 with the
// records broadcast by DPP row_newbcast (4.5 cycles an operand against 2.5).
// 6,000 x 6,000 full covariances: 22 us against 66 (160 listed of 6,000; a chain
// of dependent loads).  Scalar loads of the listed records (each wave at its own
// addresses) were bound by the scalar cache's misses, 145 cycles per record
// and CU: 1.86 ms at 200K.
constexpr int kCap = 128;  // list entries per wave (whole groups at a time)
constexpr int kNearBlock = 512;
constexpr int kNearWaves = kNearBlock / 64;
constexpr int kRows = 4, kQuads = 16;  // boxes of 16 and of 4 stationary points
// LDS for the bits: 2^18 points (32 KiB); larger clouds go window by window.
constexpr int kWinGroups = 4096;

// Tiles are (stationary block, part) pairs.  With xcd_map set they lie on a
// 1-D grid mapped XCD-aware: workgroups are dispatched to the 8 XCDs
// round-robin, so XCD x runs workgroups x, x + 8, ...; each XCD takes a
// contiguous eighth of the stationary blocks, whose near streamed points are
// about an eighth of that cloud and stay in its L2.
// Without xcd_map (clouds that fit one L2 anyway) the grid is 2-D.
constexpr int kXcds = 8;
constexpr size_t kXcdMapBytes = size_t(4) << 20;  // both clouds' records beyond one XCD's L2 (4 MiB)
__device__ __forceinline__ bool xcd_tile(int pblocks, int qsplit, int xcd_map, int *sb, int *qc) {
  if (!xcd_map) {
    *sb = blockIdx.x;
    *qc = blockIdx.y;
    return true;
  }
  const int g = blockIdx.x;
  const int bpx = (pblocks + kXcds - 1) / kXcds;
  const int xcd = g % kXcds, local = g / kXcds;
  *sb = xcd * bpx + local % bpx;
  *qc = local / bpx;
  return *sb < pblocks && *qc < qsplit;
}
static inline dim3 tile_grid(int pblocks, int qsplit, int xcd_map) {
  return xcd_map ? dim3(kXcds * ((pblocks + kXcds - 1) / kXcds) * qsplit) : dim3(pblocks, qsplit);
}

struct NearArg {
  const int *ordP;    // stationary points' Hilbert order
  const float *lamP;  // and their lam (times lam_scale: bound for the transformed ones)
  float lam_scale;
  const int *ordQ;    // streamed points' index
  const QAux *auxQ;
  const QBox *boxQ;
  int nP, nQ, pblocks, qsplit, xcd_map;
  int qchunk, gpc, ngroups;  // groups: gpc per chunk of qchunk streamed points
  int win;                   // groups per window
};

// The FP32 sums of a group go to the FP64 ones.
template <int NA>
__device__ __forceinline__ void flush_group(float *acc, double *dacc) {
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    dacc[a] += (double)acc[a];
    acc[a] = 0.0f;
  }
}

// Inclusive prefix sum over the 64 lanes (DPP: within rows of 16, then row 0's
// and 2's totals to the next row, then rows 0 and 1's to rows 2 and 3).
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ int wave_scan(int v) {
  v = dpp_add<0x111, 0xF>(v);  // row_shr:1
  v = dpp_add<0x112, 0xF>(v);  // row_shr:2
  v = dpp_add<0x114, 0xF>(v);  // row_shr:4
  v = dpp_add<0x118, 0xF>(v);  // row_shr:8
  v = dpp_add<0x142, 0xA>(v);  // row_bcast:15
  return dpp_add<0x143, 0xC>(v);  // row_bcast:31
}

// The pairs of the set bits of the lanes' groups (lane's group: 64 bits, first
// streamed point js), group by group in lane order: listed in rounds of whole
// groups, at most kCap entries (a group has at most 64).
template <class Rec, int MODE, int COMP, int NA>
__device__ __forceinline__ void walk_groups(const Rec &p, const Rec *__restrict__ Q, unsigned *list,
                                            LdsRecs<Rec, COMP> &recs, int lane, unsigned mlo, unsigned mhi, int js,
                                            double *dacc) {
  const int cnt = __popc(mlo) + __popc(mhi);
  const int incl = wave_scan(cnt), excl = incl - cnt;
  const int total = __builtin_amdgcn_readlane(incl, 63);
  for (int done = 0; done < total;) {
    const bool in = cnt > 0 && excl >= done && incl - done <= kCap;
    if (in) {
      unsigned *e = list + (excl - done);
      unsigned flag = 1u << 31;  // opens a group
      for (unsigned m = mlo; m; m &= m - 1) {
        *e++ = (unsigned)(js + __builtin_ctz(m)) | flag;
        flag = 0u;
      }
      for (unsigned m = mhi; m; m &= m - 1) {
        *e++ = (unsigned)(js + 32 + __builtin_ctz(m)) | flag;
        flag = 0u;
      }
    }
    const int last = 63 - __builtin_clzll(__ballot(in));
    const int n = __builtin_amdgcn_readlane(incl, last) - done;
    done += n;
    wave_lds_fence();
    float acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] = 0.0f;
    for (int e0 = 0; e0 < n; e0 += 64) {
      const unsigned e = list[min(e0 + lane, n - 1)];
      recs.put(lane, Q[e & 0x7fffffffu]);
      unsigned long long first = __ballot((int)e < 0);
      if (e0 == 0) first &= ~1ull;  // the sums are 0
      wave_lds_fence();
      const int m = min(64, n - e0);
      int j = 0;
      // records in flight: as many as the registers allow
      constexpr int U = RecTraits<Rec>::FULL ? (RecTraits<Rec>::D == 3 ? 1 : 2) : MODE == kModeHess ? 2 : 4;
      for (; j + U <= m; j += U) {
        Rec q[U];
#pragma unroll
        for (int k = 0; k < U; ++k) q[k] = recs.get(j + k);
#pragma unroll
        for (int k = 0; k < U; ++k) {
          if ((first >> (j + k)) & 1) flush_group<NA>(acc, dacc);
          pair_eval<MODE, COMP>(p, q[k], acc);
        }
      }
      for (; j < m; ++j) {
        if ((first >> j) & 1) flush_group<NA>(acc, dacc);
        pair_eval<MODE, COMP>(p, recs.get(j), acc);
      }
      wave_lds_fence();
    }
    flush_group<NA>(acc, dacc);
    wave_lds_fence();
  }
}

// One chunk of the Hessian pass is done: its energy and pose gradient go to r,
// EW, B (FP32, as summed) and x' - t to the point's record of this chunk, and
// the sums start again.  The transformed sources are stationary, so d = x' - y
// flips the sign of EW and, for pose_contrib, of B (see the epilogue).
constexpr int kHessRec = 12;
template <class Rec, int NA>
__device__ __forceinline__ void hess_chunk(const Rec &p, double *dacc, const double *t, double *r,
                                           float *__restrict__ out, int pi) {
  using Tr = RecTraits<Rec>;
  dacc[0] *= Tr::ESCALE;
#pragma unroll
  for (int a = 1; a < NA; ++a) dacc[a] *= -Tr::GSCALE;
  if (pi >= 0) {
    pose_contrib(p, dacc, t, r);
    float v[kHessRec];
#pragma unroll
    for (int u = 1; u < 4; ++u) v[u - 1] = -(float)dacc[u];
    // isotropic records: B = P - Q I
    const float qd = Tr::FULL ? 0.0f : (float)dacc[NA - 1];
#pragma unroll
    for (int u = 4; u < 10; ++u)
      v[u - 1] = Tr::FULL ? -(float)dacc[u] : -((float)dacc[u] - ((u == 4 || u == 7 || u == 9) ? qd : 0.0f));
    v[9] = (float)((double)p.hx + (double)p.lx - t[0]);
    v[10] = (float)((double)p.hy + (double)p.ly - t[1]);
    v[11] = (float)((double)p.hz + (double)p.lz - t[2]);
    float4 *o = reinterpret_cast<float4 *>(out + (size_t)pi * kHessRec);
#pragma unroll
    for (int q = 0; q < 3; ++q) o[q] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
  }
#pragma unroll
  for (int a = 0; a < NA; ++a) dacc[a] = 0.0;
}

// The Hessian entries of one tile -- 256 T stationary points, in kept order, of
// one chunk -- summed as the point records say: FP32 over a wave's 64 T points,
// then FP64.  Workgroup g takes tiles g, g + gridDim.x, ... and writes its 21
// sums to out.
__global__ __launch_bounds__(kBlock) void k_hess_tiles(const float *__restrict__ rec, int nP, int T, int tiles_p,
                                                       int tiles, double *__restrict__ out) {
  __shared__ float hred[kBlock / 64][21];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double sum = 0.0;
  for (int tl = blockIdx.x; tl < tiles; tl += gridDim.x) {
    const int c = tl / tiles_p, pb = tl - c * tiles_p;
    const int base = pb * (kBlock * T) + wave * (64 * T) + lane;
    float h[21];
#pragma unroll
    for (int q = 0; q < 21; ++q) h[q] = 0.0f;
    for (int k = 0; k < T; ++k) {
      const int pi = base + 64 * k;
      if (pi >= nP) continue;
      const float4 *v = reinterpret_cast<const float4 *>(rec + ((size_t)c * nP + pi) * kHessRec);
      const float4 u0 = v[0], u1 = v[1], u2 = v[2];
      const float a[10] = {0.0f, u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w, u2.x};
      const float z[3] = {u2.y, u2.z, u2.w};
      int q = 0;
#pragma unroll
      for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = i; j < 6; ++j) h[q++] += point_hessian_entry(i, j, z, a);
    }
    __syncthreads();  // the last tile's sums have been read
#pragma unroll
    for (int q = 0; q < 21; ++q) {
      const float v = wave_sum_f(h[q]);
      if (lane == 0) hred[wave][q] = v;
    }
    __syncthreads();
    if (threadIdx.x < 21) {
#pragma unroll
      for (int w = 0; w < kBlock / 64; ++w) sum += (double)hred[w][threadIdx.x];
    }
  }
  if (threadIdx.x < 21) out[(size_t)blockIdx.x * kHessPart + threadIdx.x] = sum;
}

template <class Rec>
__device__ __forceinline__ void stat_pos(const Rec &r, float *x) {
  x[0] = r.hx;
  x[1] = r.hy;
  if constexpr (RecTraits<Rec>::D == 3)
    x[2] = r.hz;
  else
    x[2] = 0.0f;
}

template <class Rec, int MODE, int COMP, bool XSRC>
__global__ __launch_bounds__(kNearBlock) __attribute__((amdgpu_waves_per_eu(MODE == kModeHess || (MODE != kModeEnergy && RecTraits<Rec>::FULL) ? 6 : 8, 8))) void k_near(
    const void *__restrict__ Pv, const Rec *__restrict__ Q, NearArg na, PoseArg ps, double *__restrict__ out,
    float *__restrict__ hess) {
  using Tr = RecTraits<Rec>;
  constexpr int D = Tr::D;
  constexpr bool GRAD = MODE != kModeEnergy;
  // the Hessian pass needs B: isotropic records then hold it in two parts
  // (the pose pass needs no G)
  constexpr int NA = MODE == kModeHess                ? (Tr::FULL ? Tr::NACC : 11)
                     : MODE == kModePose && !Tr::FULL ? 1 + D
                     : GRAD                           ? Tr::NACC
                                                      : 1;
  // per wave 64 records and kCap list entries, then the window's groups, 64
  // bits each; later the epilogue's staging
  using Recs = LdsRecs<Rec, COMP>;
  extern __shared__ __attribute__((aligned(16))) unsigned s_dyn[];
  unsigned *const s_list = s_dyn + kNearWaves * (sizeof(Recs) / 4);
  unsigned *const s_bits = s_list + kNearWaves * kCap;
  __shared__ Rec s_p[64];
  __shared__ QBox s_row[kRows], s_quad[kQuads];
  int sb, qc;
  if (!xcd_tile(na.pblocks, na.qsplit, na.xcd_map, &sb, &qc)) return;  // grid padding (whole workgroup)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ppos = sb * 64 + lane;  // Hilbert position of the lane's point
  const bool valid = ppos < na.nP;
  // the wave's first boxes, on their way while wave 0 prepares the stationary
  // points: boxes are dealt to the waves one by one (near ones follow each other)
  const int nbox = (na.nQ + 63) >> 6;
  const QBox box0 = na.boxQ[min(wave + lane * kNearWaves, nbox - 1)];

  if (wave == 0) {
    const int pp = min(ppos, na.nP - 1);
    const int pi = na.ordP[pp];
    Rec r;
    if constexpr (XSRC)
      transform_rec(reinterpret_cast<const double *>(Pv) + (size_t)pi * (D + D * D), ps, r);
    else
      r = reinterpret_cast<const Rec *>(Pv)[pi];
    s_p[lane] = r;
    float x[3];
    stat_pos(r, x);
    QBox b, b4;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float lo4 = quad_min(x[a]), hi4 = quad_max(x[a]);
      const float lo = row_min(x[a]), hi = row_max(x[a]);
      const float slack = 2.4e-7f * fmaxf(fabsf(lo), fabsf(hi));  // the lo parts
      b.lo[a] = lo - slack;
      b.hi[a] = hi + slack;
      b4.lo[a] = lo4 - slack;
      b4.hi[a] = hi4 + slack;
    }
    const float lam = na.lamP[pp] * na.lam_scale;
    b.lam = row_max(lam);
    b4.lam = quad_max(lam);
    b.pad = b4.pad = 0.0f;
    if ((lane & 3) == 0) s_quad[lane >> 2] = b4;
    if ((lane & 15) == 0) s_row[lane >> 4] = b;
  }

  Rec p;
  double dacc[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) dacc[a] = 0.0;
  double r[kPosePart];  // [E, rotation, translation]
#pragma unroll
  for (int a = 0; a < kPosePart; ++a) r[a] = 0.0;

  unsigned *const list = s_list + wave * kCap;
  Recs &recs = reinterpret_cast<Recs *>(s_dyn)[wave];
  for (int w0 = 0; w0 < na.ngroups; w0 += na.win) {
    const int wn = min(na.win, na.ngroups - w0);
    if (w0 > 0) __syncthreads();  // the last window's bits have been read
    for (int i = threadIdx.x; i < 2 * wn; i += kNearBlock) s_bits[i] = 0u;
    __syncthreads();
    if (w0 == 0) p = s_p[lane];
    for (int b0 = wave; b0 < nbox; b0 += kNearBlock) {
      const int bl = b0 + lane * kNearWaves;
      bool hit = false;
      if (bl < nbox) {
        QBox q = box0;
        if (b0 >= kNearBlock || w0 > 0) q = na.boxQ[bl];
#pragma unroll
        for (int k = 0; k < kRows; ++k)
          hit = hit || box_near(s_row[k], q.lo[0], q.lo[1], q.lo[2], q.hi[0], q.hi[1], q.hi[2], q.lam);
      }
      for (unsigned long long m = __ballot(hit); m; m &= m - 1) {
        asm volatile("" ::: "memory");
        const int i = (b0 + __builtin_ctzll(m) * kNearWaves) * 64 + lane;
        if (i >= na.nQ) continue;
        const QAux q = na.auxQ[i];
        const int j = na.ordQ[i];
        unsigned rows = 0;
#pragma unroll
        for (int k = 0; k < kRows; ++k)
          rows |= box_near(s_row[k], q.x, q.y, q.z, q.x, q.y, q.z, q.lam) ? 1u << k : 0u;
        bool near = false;
        asm volatile("" ::: "memory");  // the boxes stay in LDS (hoisted, their 160 words would spill)
        if (rows)
#pragma unroll
          for (int k = 0; k < kQuads; ++k) near = near || box_near(s_quad[k], q.x, q.y, q.z, q.x, q.y, q.z, q.lam);
        if (!near) continue;
        const int c = j / na.qchunk, r = j - c * na.qchunk;
        const int g = c * na.gpc + (r >> 6) - w0;
        if (g >= 0 && g < wn) atomicOr(&s_bits[2 * g + ((r >> 5) & 1)], 1u << (r & 31));
      }
    }
    __syncthreads();
    if constexpr (MODE == kModeHess) {
      // chunk c goes whole to part c % qsplit, wave (c / qsplit) % 8; its
      // sums leave for k_hess_tiles when its last group is done
      const int gend = w0 + wn;
      for (int c = na.qsplit * wave + qc; c * na.gpc < gend; c += na.qsplit * kNearWaves) {
        if ((c + 1) * na.gpc <= w0) continue;
        const int c1 = min((c + 1) * na.gpc, gend);
        for (int gb = max(c * na.gpc, w0); gb < c1; gb += 64) {
          const int g = gb + lane;
          const bool own = g < c1;
          walk_groups<Rec, MODE, COMP, NA>(p, Q, list, recs, lane, own ? s_bits[2 * (g - w0)] : 0u,
                                           own ? s_bits[2 * (g - w0) + 1] : 0u,
                                           c * na.qchunk + (g - c * na.gpc) * 64, dacc);
        }
        if ((c + 1) * na.gpc > gend) break;  // goes on in the next window
        hess_chunk<Rec, NA>(p, dacc, ps.t, r, hess + (size_t)c * na.nP * kHessRec, valid ? na.ordP[ppos] : -1);
      }
    } else {
      // group g goes to part g % qsplit, wave (g / qsplit) % 8
      for (int g0 = 0; g0 < wn; g0 += kNearBlock * na.qsplit) {
        const int g = g0 + (lane * kNearWaves + wave) * na.qsplit + qc;
        const bool own = g < wn;
        const int c = (w0 + g) / na.gpc;
        walk_groups<Rec, MODE, COMP, NA>(p, Q, list, recs, lane, own ? s_bits[2 * g] : 0u, own ? s_bits[2 * g + 1] : 0u,
                                         c * na.qchunk + (w0 + g - c * na.gpc) * 64, dacc);
      }
    }
  }

  // Isotropic records: variances were times ln 4 (ESCALE, GSCALE).  A pose
  // pass with COMP 2 has the transformed sources stationary: d = x' - y
  // flips the sign of EW (and of nothing else: B holds d d^T), and the
  // gradient is then taken about the sources, whose rotation also turns
  // their covariances.  With EW and B both negated, pose_contrib's
  // (p - t) x EW + vee(S_p B - B S_p) is exactly that gradient.
  constexpr bool kSwapped = MODE == kModePose && COMP == 2;
  if (MODE != kModeHess && (!RecTraits<Rec>::FULL || kSwapped)) {
    constexpr double gs = kSwapped ? -RecTraits<Rec>::GSCALE : RecTraits<Rec>::GSCALE;
    dacc[0] *= RecTraits<Rec>::ESCALE;
#pragma unroll
    for (int a = 1; a < NA; ++a) dacc[a] *= gs;
  }

  double *stage = reinterpret_cast<double *>(s_dyn);
  if constexpr (MODE == kModePoint) {
    // the 8 waves' sums of each point, in wave order, kHalf values at a time
    constexpr int kHalf = (NA + 1) / 2;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int nv = h == 0 ? kHalf : NA - kHalf;
      __syncthreads();
#pragma unroll
      for (int a = 0; a < nv; ++a) stage[(wave * kHalf + a) * 64 + lane] = dacc[h * kHalf + a];
      __syncthreads();
      for (int e = threadIdx.x; e < 64 * nv; e += kNearBlock) {
        const int k = e / nv, a = e - k * nv;
        if (sb * 64 + k < na.nP) {
          double s = stage[a * 64 + k];
#pragma unroll
          for (int w = 1; w < kNearWaves; ++w) s += stage[(w * kHalf + a) * 64 + k];
          out[((size_t)qc * na.nP + na.ordP[sb * 64 + k]) * NA + h * kHalf + a] = s;
        }
      }
    }
    return;
  }

  if (MODE != kModeHess && valid) {
    if constexpr (GRAD)
      pose_contrib(p, dacc, ps.t, r);
    else
      r[0] += dacc[0];
  }
  double *o = out + ((size_t)qc * na.pblocks + sb) * kPosePart;
  __syncthreads();  // the bits have been read
  if (GRAD) {
    // Workgroup sums of the kPosePart values in a fixed order: every lane's
    // values go to LDS; wave a adds entries lane, lane + 64, ... of value a
    // (consecutive lanes read consecutive doubles: no bank conflict), then
    // sums over its lanes by DPP.
    static_assert(kPosePart == kNearWaves, "one wave per pose value");
#pragma unroll
    for (int a = 0; a < kPosePart; ++a) stage[a * kNearBlock + threadIdx.x] = r[a];
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < kNearWaves; ++i) s += stage[wave * kNearBlock + lane + 64 * i];
    s = wave_sum(s);
    if (lane == 0) o[wave] = s;
  } else {
    const double v = wave_sum(r[0]);
    if (lane == 0) stage[wave] = v;
    __syncthreads();
    if (threadIdx.x < kPosePart) {
      double s = 0.0;
      if (threadIdx.x == 0) {
        s = stage[0];
#pragma unroll
        for (int w = 1; w < kNearWaves; ++w) s += stage[w];
      }
      o[threadIdx.x] = s;
    }
  }
}

// Fixed-order sum of the per-workgroup partials over kRedGroups workgroups
// at most: workgroup g sums the contiguous range [g len, (g + 1) len) --
// thread t adds partials t, t + 256, ... of it, then the 256 lanes' values
// are summed through LDS and half-wave sums as in the pair kernel -- and
// writes its kPosePart sums to res[kPosePart g, ...), the context's pinned
// host slots; the host adds the workgroups' sums in order.
constexpr int kRedGroups = 8;
__global__ __launch_bounds__(kBlock) void k_reduce_parts(
    const double *__restrict__ parts, int nparts, double *__restrict__ res) {
  const int len = (nparts + (int)gridDim.x - 1) / (int)gridDim.x;
  const int q0 = blockIdx.x * len, q1 = min(q0 + len, nparts);
  double s[kPosePart];
#pragma unroll
  for (int a = 0; a < kPosePart; ++a) s[a] = 0.0;
  for (int q = q0 + (int)threadIdx.x; q < q1; q += kBlock) {
    const double4 *p = reinterpret_cast<const double4 *>(parts + (size_t)q * kPosePart);
    const double4 u = p[0], v = p[1];
    s[0] += u.x; s[1] += u.y; s[2] += u.z; s[3] += u.w;
    s[4] += v.x; s[5] += v.y; s[6] += v.z; s[7] += v.w;
  }
  __shared__ double stage[kPosePart][kBlock];
#pragma unroll
  for (int a = 0; a < kPosePart; ++a) stage[a][threadIdx.x] = s[a];
  __syncthreads();
  const int a = threadIdx.x >> 5, k = threadIdx.x & 31;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double t = 0.0;
#pragma unroll
  for (int i = 0; i < kBlock / 32; ++i) t += stage[a][k + 32 * i];
  double lo, hi;
  half_wave_sums(t, lo, hi);
  if (lane == 0) {
    res[kPosePart * blockIdx.x + 2 * wave] = lo;
    res[kPosePart * blockIdx.x + 2 * wave + 1] = hi;
  }
}

// The 21 Hessian sums of k_hess_tiles' workgroups (kHessPart doubles each), in a
// fixed order: thread (a, k) adds records k, k + 32, ... of entry a, then each
// half wave sums its 32.
constexpr int kHessGroups = 512;
__global__ __launch_bounds__(1024) void k_reduce_hess(const double *__restrict__ parts, int nparts,
                                                      double *__restrict__ res) {
  const int a = threadIdx.x & 31, k = threadIdx.x >> 5;
  __shared__ double stage[32][33];
  double s = 0.0;
  if (a < 21)
    for (int q = k; q < nparts; q += 32) s += parts[(size_t)q * kHessPart + a];
  stage[a][k] = s;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double lo, hi;
  half_wave_sums(stage[2 * wave + (lane >> 5)][lane & 31], lo, hi);
  if (lane == 0 && 2 * wave < 21) res[2 * wave] = lo;
  if (lane == 0 && 2 * wave + 1 < 21) res[2 * wave + 1] = hi;
}

// Per-point sums over streamed chunks, in chunk order.
__global__ __launch_bounds__(kBlock) void k_reduce_points(
    const double *__restrict__ parts, int nP, int nchunks, int nacc,
    double *__restrict__ res) {
  const size_t idx = (size_t)blockIdx.x * kBlock + threadIdx.x;
  const size_t total = (size_t)nP * nacc;
  if (idx >= total) return;
  double s = 0.0;
  for (int c = 0; c < nchunks; ++c) s += parts[(size_t)c * total + idx];
  res[idx] = s;
}

// ---------------------------------------------------------------------------
// Launch planning
// ---------------------------------------------------------------------------
struct Plan {
  // Sub-tiles: chunks of qchunk streamed points, each cut into groups of kSub
  // from its start.  They fix how the FP32 sums are grouped.
  int qchunk = 1, gpc = 1, ngroups = 1;
  int T = 1, tiles_p = 1, qchunks = 1;  // chunk tiles: tiles_p times 256 T stationary points, qchunks chunks
  // Launch: pblocks workgroups of 64 stationary points times qsplit parts of
  // the groups.
  int pblocks = 1, qsplit = 1;
};

static int env_int(const char *name, int dflt) {
  const char *v = getenv(name);
  return (v && *v) ? atoi(v) : dflt;
}

// Waves a launch aims at when the stationary points alone give fewer: 4 per
// SIMD of the 256 CUs.
constexpr int kLaunchWaves = 4096;

// Chunks so that tiles of 256 T stationary points x one chunk make about
// target_waves waves, each chunk at least kMinChunk points.
static Plan make_plan(int nP, int nQ, int mode, int T, int target_waves, int launch_waves, int max_chunks = 64) {
  Plan pl;
  const int tiles_p = (nP + kBlock * T - 1) / (kBlock * T);
  const int waves_p = tiles_p * (kBlock / 64);
  int qc = (target_waves + waves_p - 1) / waves_p;
  int maxc = (nQ + kMinChunk - 1) / kMinChunk;
  if (mode == kModePoint) maxc = std::min(maxc, max_chunks);
  maxc = std::min({maxc, 65535, (int)(INT32_MAX / kBlock / (tiles_p + kXcds))});
  qc = std::max(1, std::min(qc, maxc));
  pl.qchunk = (nQ + qc - 1) / qc;
  pl.T = T;
  pl.tiles_p = tiles_p;
  pl.qchunks = (nQ + pl.qchunk - 1) / pl.qchunk;
  pl.gpc = (pl.qchunk + kSub - 1) / kSub;
  pl.ngroups = pl.qchunks * pl.gpc;
  pl.pblocks = (nP + 63) / 64;
  const int waves = pl.pblocks * kNearWaves;
  pl.qsplit = std::max(1, std::min((launch_waves + waves - 1) / waves, (pl.ngroups + kNearWaves - 1) / kNearWaves));
  return pl;
}

// Sub-tiles: T = 2 and 4096 waves, 16384 for very large problems (environment
// overrides).  Launch: kLaunchWaves, or what dugma_autotune chose.
static Plan ctx_plan(const dugma_ctx *c, int nP, int nQ, int mode, bool iso) {
  int T = 2, tw = ((double)nP * nQ >= 1e9) ? 16384 : 4096;
  T = env_int("DUGMA_LANE_POINTS", T) == 1 ? 1 : 2;
  tw = env_int("DUGMA_TARGET_WAVES", tw);
  const dugma_ctx::Tuned &tu = c->tuned[mode == kModeEnergy ? 0 : 1][iso ? 1 : 0];
  return make_plan(nP, nQ, mode, T, tw, tu.target_waves > 0 ? tu.target_waves : kLaunchWaves);
}

// A pass's two point sets: the stationary cloud is 0 (targets) or 1
// (sources), the other one is streamed.
struct Sets {
  int stat;        // stationary cloud
  const void *P;   // its records in kept order (null: transformed from the source data in the kernel)
  const void *Q;   // streamed records in kept order
  float lam_scale;
};

template <class Rec, int MODE, int COMP, bool XSRC>
static void launch_near_x(dugma_ctx *c, const Plan &pl, const Sets &st, const PoseArg &ps, double *out,
                          float *hess = nullptr) {
  NearArg na;
  const int nP = st.stat == 0 ? c->nT : c->nS, nQ = st.stat == 0 ? c->nS : c->nT;
  const NearCloud &cp = c->near[st.stat], &cq = c->near[1 - st.stat];
  na.ordP = cp.ord;
  na.lamP = cp.lam;
  na.lam_scale = st.stat == 0 ? 1.0f : st.lam_scale;
  na.ordQ = cq.ord;
  na.auxQ = cq.aux;
  na.boxQ = cq.box;
  na.nP = nP;
  na.nQ = nQ;
  na.pblocks = pl.pblocks;
  na.qsplit = pl.qsplit;
  // the XCD tile order for clouds beyond one L2; DUGMA_XCD_ORDER=0 in the
  // environment keeps the 2-D order (the sums are the same, bit for bit)
  na.xcd_map = (size_t)(nP + nQ) * sizeof(Rec) > kXcdMapBytes && env_int("DUGMA_XCD_ORDER", 1) != 0 ? 1 : 0;
  na.qchunk = pl.qchunk;
  na.gpc = pl.gpc;
  na.ngroups = pl.ngroups;
  // windows of whole chunks for the Hessian pass (or parts of one chunk)
  na.win = MODE == kModeHess && pl.gpc <= kWinGroups ? kWinGroups / pl.gpc * pl.gpc : kWinGroups;
  constexpr size_t kStage = MODE == kModeEnergy ? sizeof(double) * kNearWaves
                            : MODE == kModePoint ? sizeof(double) * kNearBlock * ((RecTraits<Rec>::NACC + 1) / 2)
                                                 : sizeof(double) * kNearBlock * kPosePart;
  const size_t lds =
      std::max(kStage, kNearWaves * (sizeof(LdsRecs<Rec, COMP>) + sizeof(unsigned) * kCap) +
                           (size_t)8 * std::min(pl.ngroups, kWinGroups));
  const void *P = XSRC ? (const void *)c->dSsrc : st.P;
  hipLaunchKernelGGL((k_near<Rec, MODE, COMP, XSRC>), tile_grid(pl.pblocks, pl.qsplit, na.xcd_map),
                     dim3(kNearBlock), lds, c->stream, P, (const Rec *)st.Q, na, ps, out, hess);
}

// comp: 0 none, 1 streamed side carries the lo part, 2 stationary side does.
template <class Rec>
static void launch_near(dugma_ctx *c, int mode, int comp, const Plan &pl, const Sets &st, const PoseArg &ps,
                        double *out) {
#define DUGMA_L(M, C, X) launch_near_x<Rec, M, C, X>(c, pl, st, ps, out)
  if (mode == kModeEnergy) {
    // comp 2 in these passes: the transformed sources are stationary (see pose_pass)
    if (comp == 2) DUGMA_L(kModeEnergy, 2, true); else if (comp == 1) DUGMA_L(kModeEnergy, 1, false); else DUGMA_L(kModeEnergy, 0, false);
  } else if (mode == kModePose) {
    if (comp == 2) DUGMA_L(kModePose, 2, true); else if (comp == 1) DUGMA_L(kModePose, 1, false); else DUGMA_L(kModePose, 0, false);
  } else {
    if (comp == 1) DUGMA_L(kModePoint, 1, false);
    else if (comp == 2) DUGMA_L(kModePoint, 2, false);
    else DUGMA_L(kModePoint, 0, false);
  }
#undef DUGMA_L
}

// Device data are in scaled units: positions times s = 2^k, covariances
// times s^2 (chosen at init so covariances are O(1)); exact in binary FP.
static PoseArg make_pose(const dugma_ctx *c, const double *R, const double *t) {
  PoseArg ps;
  memset(&ps, 0, sizeof(ps));
  for (int a = 0; a < c->D * c->D; ++a) ps.R[a] = R[a];
  for (int a = 0; a < c->D; ++a) ps.t[a] = t[a] * c->scale;
  return ps;
}

// The transformed sources' records in kept order, with their index: for the
// passes that stream them.
static int transform_sources(dugma_ctx *c, const PoseArg &ps, bool iso, float lam_scale) {
  if (c->nS == 0) return DUGMA_OK;
  dim3 grid((c->nS + kBlock - 1) / kBlock), block(kBlock);
  void *out = iso ? c->dSrecI : c->dSrecF;
#define DUGMA_T(R) hipLaunchKernelGGL(k_transform_src<R>, grid, block, 0, c->stream, c->dSsrc, c->nS, ps, (R *)out)
  if (c->D == 3) {
    if (iso) DUGMA_T(Rec3I); else DUGMA_T(Rec3F);
  } else {
    if (iso) DUGMA_T(Rec2I); else DUGMA_T(Rec2F);
  }
#undef DUGMA_T
  DUGMA_HIP(hipGetLastError());
  return near_index_sources(c, iso, out, lam_scale);
}

// Bound of R's largest singular value squared (1 for a rotation): what R can
// do to a covariance's largest eigenvalue.  Infinite (every pair counts) for an R
// so far from a similarity that it also spoils a covariance's conditioning.
static float pose_lam_scale(int D, const double *R) {
  double big = 0.0, small = INFINITY;
  for (int a = 0; a < D; ++a) {
    double row = 0.0, diag = 0.0;
    for (int b = 0; b < D; ++b) {
      double v = 0.0;
      for (int k = 0; k < D; ++k) v += R[k + D * a] * R[k + D * b];
      row += std::fabs(v);
      if (a == b) diag = v;
    }
    big = std::max(big, row);
    small = std::min(small, 2.0 * diag - row);
  }
  return small > 0.25 * big ? (float)(big * 1.000001) : INFINITY;
}

static int resolve_iso(dugma_ctx *c, int cov_mode, bool *iso) {
  if (cov_mode == DUGMA_COV_FULL) {
    *iso = false;
  } else if (cov_mode == DUGMA_COV_ISO) {
    if (!c->iso) return fail(DUGMA_ERR_ARG, "DUGMA_COV_ISO: covariances are not all isotropic");
    *iso = true;
  } else if (cov_mode == DUGMA_COV_AUTO) {
    *iso = c->iso;
  } else {
    return fail(DUGMA_ERR_ARG, "unknown cov_mode");
  }
  return DUGMA_OK;
}

static double gauss_norm(int D) {
  const double two_pi = 6.283185307179586476925;
  return D == 3 ? 1.0 / (two_pi * std::sqrt(two_pi)) : 1.0 / two_pi;
}

static bool comp_enabled() { return env_int("DUGMA_COMPENSATED", 1) != 0; }
// the pose and energy passes keep the transformed sources stationary unless
// DUGMA_STATIONARY_SOURCES=0 (then the targets, with the lo correction on
// the streamed side); both give the same sums to FP32 rounding
static bool sources_stationary() { return comp_enabled() && env_int("DUGMA_STATIONARY_SOURCES", 1) != 0; }

// Energy-only or fused pose pass; res receives [E, rotation, translation]
// in caller units.
static int pose_pass(dugma_ctx *c, const double *R, const double *t, bool iso,
                     int mode, double *res, double *fixed_parts = nullptr, size_t fixed_records = 0) {
  const int D = c->D;
  const int width = mode == kModeEnergy ? 1 : (D == 3 ? 7 : 4);
  for (int a = 0; a < width; ++a) res[a] = 0.0;
  if (c->nT == 0 || c->nS == 0) return DUGMA_OK;
  // everything the launches need is settled first, so that they leave the
  // host back to back
  PoseArg ps = make_pose(c, R, t);
  // The passes keep the transformed sources (FP32 hi + lo) stationary and
  // stream the targets (exact in FP32): the lo correction is then an
  // operation on VGPRs only (COMP 2) instead of a second one on the streamed
  // SGPRs (COMP 1), and the kernel transforms its own 64 sources.  E is
  // symmetric in the two roles; the gradient sums change sign (kernel
  // epilogue).  Without compensation the targets stay stationary (COMP 0).
  const bool swap = sources_stationary();
  const int comp = swap ? 2 : (comp_enabled() ? 1 : 0);
  Plan pl = swap ? ctx_plan(c, c->nS, c->nT, mode, iso) : ctx_plan(c, c->nT, c->nS, mode, iso);
  const size_t nparts = (size_t)pl.pblocks * pl.qsplit;
  // few partials: the pair kernel writes them to pinned host memory and the
  // host sums them as they arrive; many: a device reduction launch
  const bool host_sum = nparts <= (size_t)dugma_ctx::kHostParts;
  double *parts = c->dparts;
  int rc;
  if (fixed_parts && std::max((size_t)pl.tiles_p * pl.qchunks, nparts) > fixed_records)
    return fail(DUGMA_ERR_SIZE, "dugma_energy_grad_noalloc: the launch needs more partial records than the "
                                "scratch array holds (lower DUGMA_TARGET_WAVES or the autotuned wave count)");
  if (!host_sum && fixed_parts) {
    parts = fixed_parts;
  } else if (!host_sum) {
    rc = c->part.ensure(nparts * kPosePart * sizeof(double));
    if (rc) return rc;
    parts = (double *)c->part.ptr;
  }
  const int groups = (int)std::min<size_t>(kRedGroups, (nparts + kBlock - 1) / kBlock);
  const float lam_scale = pose_lam_scale(D, R);
  if (host_sum)
    preset_slots(c->hparts, (int)(kPosePart * nparts));
  else
    preset_slots(c->hres, kPosePart * groups);
  if (!swap) {
    rc = transform_sources(c, ps, iso, lam_scale);
    if (rc) return rc;
  }
  PairTimer timer(c);
  const void *tgt = iso ? c->dTrecI : c->dTrecF, *src = iso ? c->dSrecI : c->dSrecF;
  const Sets st = {swap ? 1 : 0, swap ? nullptr : tgt, swap ? tgt : src, lam_scale};
  if (D == 3) {
    if (iso)
      launch_near<Rec3I>(c, mode, comp, pl, st, ps, parts);
    else
      launch_near<Rec3F>(c, mode, comp, pl, st, ps, parts);
  } else {
    if (iso)
      launch_near<Rec2I>(c, mode, comp, pl, st, ps, parts);
    else
      launch_near<Rec2F>(c, mode, comp, pl, st, ps, parts);
  }
  timer.stop();
  DUGMA_HIP(hipGetLastError());
  if (!host_sum) {
    hipLaunchKernelGGL(k_reduce_parts, dim3(groups), dim3(kBlock), 0, c->stream, parts, (int)nparts, c->dres);
  }
  DUGMA_HIP(hipGetLastError());
  rc = host_sum ? wait_slots(c, c->hparts, (int)(kPosePart * nparts)) : wait_slots(c, c->hres, kPosePart * groups);
  if (rc) return rc;
  timer.finish();
  double sum[kPosePart] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (host_sum) {
    const volatile double *hp = c->hparts;
    for (size_t q = 0; q < nparts; ++q)
      for (int a = 0; a < width; ++a) sum[a] += hp[q * kPosePart + a];
  } else {
    const volatile double *hr = c->hres;
    for (int g = 0; g < groups; ++g)
      for (int a = 0; a < width; ++a) sum[a] += hr[kPosePart * g + a];
  }
  // unscale: E ~ s^D, rotation gradient ~ s^D, translation gradient ~ s^(D+1)
  const double cn = gauss_norm(D);
  const double sD = std::pow(c->scale, D);
  const int nrot = D == 3 ? 3 : 1;
  res[0] = cn * sD * sum[0];
  for (int a = 1; a < width; ++a) res[a] = cn * sD * sum[a] * (a > nrot ? c->scale : 1.0);
  return DUGMA_OK;
}

// The fused pose pass with the sums of an approximate Hessian (3-D, the
// transformed sources stationary): res = [E, rotation (3), translation
// (3)] as pose_pass gives them, H = the upper triangle, row by row, of the
// 6 x 6 Hessian of E in (w, dt) for R <- exp([w]x) R, t <- t + dt, the turn
// of the sources' covariances left out of its second order; caller units.
static int pose_hess_pass(dugma_ctx *c, const double *R, const double *t, bool iso, double *res, double *H) {
  for (int a = 0; a < 7; ++a) res[a] = 0.0;
  for (int a = 0; a < 21; ++a) H[a] = 0.0;
  if (c->D != 3) return fail(DUGMA_ERR_ARG, "the pose Hessian is 3-D only");
  if (c->nT == 0 || c->nS == 0) return DUGMA_OK;
  PoseArg ps = make_pose(c, R, t);
  const Plan pl = ctx_plan(c, c->nS, c->nT, kModePose, iso);
  const size_t nparts = (size_t)pl.pblocks * pl.qsplit;
  const int groups = (int)std::min<size_t>(kRedGroups, (nparts + kBlock - 1) / kBlock);
  const int tiles = pl.tiles_p * pl.qchunks, hgroups = std::min(tiles, kHessGroups);
  // scratch: pose partials | tile sums | per chunk and point the Hessian's inputs
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t o_tile = al(nparts * kPosePart * sizeof(double));
  const size_t o_rec = o_tile + al((size_t)hgroups * kHessPart * sizeof(double));
  int rc = c->part.ensure(o_rec + (size_t)pl.qchunks * c->nS * kHessRec * sizeof(float));
  if (rc) return rc;
  char *base = (char *)c->part.ptr;
  double *parts = (double *)base, *tsum = (double *)(base + o_tile);
  float *rec = (float *)(base + o_rec);
  double *hslots = c->hres + dugma_ctx::kResMoments;
  preset_slots(c->hres, kPosePart * groups);
  preset_slots(hslots, 21);
  PairTimer timer(c);
  const Sets st = {1, nullptr, iso ? c->dTrecI : c->dTrecF, pose_lam_scale(3, R)};
  if (iso)
    launch_near_x<Rec3I, kModeHess, 2, true>(c, pl, st, ps, parts, rec);
  else
    launch_near_x<Rec3F, kModeHess, 2, true>(c, pl, st, ps, parts, rec);
  timer.stop();
  hipLaunchKernelGGL(k_reduce_parts, dim3(groups), dim3(kBlock), 0, c->stream, parts, (int)nparts, c->dres);
  hipLaunchKernelGGL(k_hess_tiles, dim3(hgroups), dim3(kBlock), 0, c->stream, rec, c->nS, pl.T, pl.tiles_p, tiles,
                     tsum);
  hipLaunchKernelGGL(k_reduce_hess, dim3(1), dim3(1024), 0, c->stream, tsum, hgroups,
                     c->dres + dugma_ctx::kResMoments);
  DUGMA_HIP(hipGetLastError());
  rc = wait_slots(c, hslots, 21);
  if (!rc) rc = wait_slots(c, c->hres, kPosePart * groups);
  if (rc) return rc;
  timer.finish();
  double sum[kPosePart], hsum[21];
  const volatile double *hr = c->hres, *hh = hslots;
  for (int a = 0; a < kPosePart; ++a) sum[a] = 0.0;
  for (int g = 0; g < groups; ++g)
    for (int a = 0; a < kPosePart; ++a) sum[a] += hr[kPosePart * g + a];
  for (int a = 0; a < 21; ++a) hsum[a] = hh[a];
  // unscale: E ~ s^3, and a factor s per translation index
  const double cn = gauss_norm(3), sc = c->scale, sD = sc * sc * sc;
  res[0] = cn * sD * sum[0];
  for (int a = 1; a < 7; ++a) res[a] = cn * sD * sum[a] * (a > 3 ? sc : 1.0);
  int q = 0;
  for (int i = 0; i < 6; ++i)
    for (int j = i; j < 6; ++j, ++q) H[q] = cn * sD * hsum[q] * (i >= 3 ? sc : 1.0) * (j >= 3 ? sc : 1.0);
  return DUGMA_OK;
}

static int check_pose_args(dugma_ctx *c, const double *R, const double *t) {
  if (!c) return fail(DUGMA_ERR_ARG, "null context");
  if (!R || !t) return fail(DUGMA_ERR_ARG, "null R or t");
  for (int a = 0; a < c->D * c->D; ++a)
    if (!std::isfinite(R[a])) return fail(DUGMA_ERR_ARG, "R is not finite");
  for (int a = 0; a < c->D; ++a)
    if (!std::isfinite(t[a])) return fail(DUGMA_ERR_ARG, "t is not finite");
  return DUGMA_OK;
}

// Left perturbation of the pose: 3-D p = [w, dt], R <- exp([w]x) R;
// 2-D p = [theta, dt], R <- Rot(theta) R.
static void perturb(int D, const double *R, const double *t, const double *p,
                    double *Rn, double *tn) {
  if (D == 3) {
    const double *w = p;
    double th = std::sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    double A = th < 1e-12 ? 1.0 : std::sin(th) / th;
    double B = th < 1e-12 ? 0.5 : (1.0 - std::cos(th)) / (th * th);
    double K[9] = {0, w[2], -w[1], -w[2], 0, w[0], w[1], -w[0], 0};
    double E[9];
    for (int a = 0; a < 3; ++a)
      for (int c = 0; c < 3; ++c) {
        double k2 = 0;
        for (int b = 0; b < 3; ++b) k2 += K[a + 3 * b] * K[b + 3 * c];
        E[a + 3 * c] = (a == c ? 1.0 : 0.0) + A * K[a + 3 * c] + B * k2;
      }
    for (int a = 0; a < 3; ++a)
      for (int c = 0; c < 3; ++c) {
        double s = 0;
        for (int b = 0; b < 3; ++b) s += E[a + 3 * b] * R[b + 3 * c];
        Rn[a + 3 * c] = s;
      }
    for (int a = 0; a < 3; ++a) tn[a] = t[a] + p[3 + a];
  } else {
    double cs = std::cos(p[0]), sn = std::sin(p[0]);
    double E[4] = {cs, sn, -sn, cs};
    for (int a = 0; a < 2; ++a)
      for (int c = 0; c < 2; ++c)
        Rn[a + 2 * c] = E[a] * R[2 * c] + E[a + 2] * R[1 + 2 * c];
    tn[0] = t[0] + p[1];
    tn[1] = t[1] + p[2];
  }
}

// Per-point gradients on the way out: from a point's sums (NACC of point_pass)
// to the caller's units and layout -- gradient of the point (D) at P + i D, of
// its covariance (D x D, column-major) at C + i D D, i its original index -- and,
// per workgroup, kPointSums sums: [E, dE/dw (3) or dE/dtheta, dE/dt (3), dE/ddR
// (9, column-major, at identity)], the pose's of the sources only.  FP64, one
// thread per point; on the host (8 threads) the same took 1.3 ms for two
// 76,800-point clouds, here 12 us.
constexpr int kPointSums = 16;
struct PointUnits {
  double cn, gpos, gcov;  // Gaussian norm; unscaling of point and covariance gradients
};
template <int D, bool TARGET>
__global__ __launch_bounds__(kBlock) void k_points_out(const double *__restrict__ acc,
                                                       const double *__restrict__ src,
                                                       const int *__restrict__ idx, int nP, PoseArg ps,
                                                       PointUnits pu, double *__restrict__ P,
                                                       double *__restrict__ C, double *__restrict__ sums) {
  constexpr int DD = D * D, NACC = D == 3 ? kAcc3F : kAcc2F;
  const int k = blockIdx.x * kBlock + threadIdx.x;
  double s[kPointSums];
#pragma unroll
  for (int a = 0; a < kPointSums; ++a) s[a] = 0.0;
  if (k < nP) {
    double a[NACC];
#pragma unroll
    for (int q = 0; q < NACC; ++q) a[q] = acc[(size_t)k * NACC + q];
    const size_t i = (size_t)idx[k];
    double H[DD];  // dE/dS
#pragma unroll
    for (int u = 0; u < D; ++u)
#pragma unroll
      for (int v = u; v < D; ++v) {
        const int q = 1 + D + (D == 3 ? (u == 0 ? v : u == 1 ? 2 + v : 5) : u + v);
        H[u + D * v] = H[v + D * u] = 0.5 * pu.cn * a[q];
      }
    if constexpr (TARGET) {
      s[0] = a[0];
#pragma unroll
      for (int d = 0; d < D; ++d) P[i * D + d] = -pu.cn * a[1 + d] * pu.gpos;
#pragma unroll
      for (int q = 0; q < DD; ++q) C[i * DD + q] = H[q] * pu.gcov;
    } else {
      const double *x = src + (size_t)k * (D + DD);
      const double *R = ps.R;
      double g[D], p[D], RS[DD], Sp[DD];
#pragma unroll
      for (int d = 0; d < D; ++d) g[d] = -pu.cn * a[1 + d];  // dE/dx'
#pragma unroll
      for (int d = 0; d < D; ++d) {  // R x (= x' - t)
        double v = 0;
#pragma unroll
        for (int b = 0; b < D; ++b) v += R[d + D * b] * x[b];
        p[d] = v;
      }
#pragma unroll
      for (int u = 0; u < D; ++u)
#pragma unroll
        for (int c = 0; c < D; ++c) {
          double v = 0;
#pragma unroll
          for (int b = 0; b < D; ++b) v += R[u + D * b] * x[D + b + D * c];
          RS[u + D * c] = v;
        }
#pragma unroll
      for (int u = 0; u < D; ++u)
#pragma unroll
        for (int c = 0; c < D; ++c) {
          double v = 0;
#pragma unroll
          for (int b = 0; b < D; ++b) v += RS[u + D * b] * R[c + D * b];
          Sp[u + D * c] = v;
        }
      double HS[DD], SH[DD];
#pragma unroll
      for (int u = 0; u < D; ++u)
#pragma unroll
        for (int c = 0; c < D; ++c) {
          double v = 0, w = 0;
#pragma unroll
          for (int b = 0; b < D; ++b) {
            v += H[u + D * b] * Sp[b + D * c];
            w += Sp[u + D * b] * H[b + D * c];
          }
          HS[u + D * c] = v;
          SH[u + D * c] = w;
        }
      if constexpr (D == 3) {  // p x g - 2 vee(S'H - HS')
        s[1] = p[1] * g[2] - p[2] * g[1] - 2.0 * (SH[2 + 3 * 1] - HS[2 + 3 * 1]);
        s[2] = p[2] * g[0] - p[0] * g[2] - 2.0 * (SH[0 + 3 * 2] - HS[0 + 3 * 2]);
        s[3] = p[0] * g[1] - p[1] * g[0] - 2.0 * (SH[1 + 3 * 0] - HS[1 + 3 * 0]);
      } else {  // tr(H (J S' - S' J)) = tr((S'H - HS') J) = 2 (S'H - HS')_12
        s[1] = g[1] * p[0] - g[0] * p[1] + 2.0 * (SH[0 + 2 * 1] - HS[0 + 2 * 1]);
      }
#pragma unroll
      for (int d = 0; d < D; ++d) s[4 + d] = g[d];
      // dE/d dR at identity: g p^T + 2 H S'
#pragma unroll
      for (int u = 0; u < D; ++u)
#pragma unroll
        for (int c = 0; c < D; ++c) s[7 + u + D * c] = g[u] * p[c] + 2.0 * HS[u + D * c];
#pragma unroll
      for (int b = 0; b < D; ++b) {
        double v = 0;
#pragma unroll
        for (int u = 0; u < D; ++u) v += R[u + D * b] * g[u];
        P[i * D + b] = v * pu.gpos;
      }
#pragma unroll
      for (int b = 0; b < D; ++b)
#pragma unroll
        for (int c = 0; c < D; ++c) {
          double v = 0;
#pragma unroll
          for (int u = 0; u < D; ++u)
#pragma unroll
            for (int e = 0; e < D; ++e) v += R[u + D * b] * H[u + D * e] * R[e + D * c];
          C[i * DD + b + D * c] = v * pu.gcov;
        }
    }
  }
  // workgroup sums in a fixed order
  __shared__ double red[kBlock / 64][kPointSums];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int a = 0; a < (TARGET ? 1 : kPointSums); ++a) {
    const double v = wave_sum(s[a]);
    if (lane == 0) red[wave][a] = v;
  }
  __syncthreads();
  if (threadIdx.x < (TARGET ? 1 : kPointSums)) {
    double v = red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) v += red[w][threadIdx.x];
    sums[(size_t)blockIdx.x * kPointSums + threadIdx.x] = v;
  }
}

// One per-point pass (stationary cloud st.stat), full covariance records;
// writes per-point FP64 sums [nP][NACC] to out (device).
// Sub-tiles: chunks for 65,536 waves, at most 64 and 1 GiB of per-chunk sums.
constexpr size_t kPointPartBytes = size_t(1) << 30;
static int point_pass(dugma_ctx *c, const Sets &st, const PoseArg &ps, int comp, double *out) {
  const int D = c->D;
  const int nacc = D == 3 ? kAcc3F : kAcc2F;
  const int nP = st.stat == 0 ? c->nT : c->nS, nQ = st.stat == 0 ? c->nS : c->nT;
  const int max_chunks =
      (int)std::max<size_t>(1, std::min<size_t>(64, kPointPartBytes / ((size_t)nP * nacc * sizeof(double))));
  Plan pl = make_plan(nP, nQ, kModePoint, 1, env_int("DUGMA_POINT_WAVES", 65536), kLaunchWaves, max_chunks);
  double *parts = out;  // one part: the sums themselves
  if (pl.qsplit > 1) {
    int rc = c->part.ensure((size_t)pl.qsplit * nP * nacc * sizeof(double));
    if (rc) return rc;
    parts = (double *)c->part.ptr;
  }
  if (!comp_enabled()) comp = 0;
  PairTimer timer(c);
  if (D == 3)
    launch_near<Rec3F>(c, kModePoint, comp, pl, st, ps, parts);
  else
    launch_near<Rec2F>(c, kModePoint, comp, pl, st, ps, parts);
  timer.stop();
  DUGMA_HIP(hipGetLastError());
  if (pl.qsplit > 1) {
    const size_t total = (size_t)nP * nacc;
    hipLaunchKernelGGL(k_reduce_points, dim3((unsigned)((total + kBlock - 1) / kBlock)), dim3(kBlock), 0, c->stream,
                       parts, nP, pl.qsplit, nacc, out);
    DUGMA_HIP(hipGetLastError());
  }
  timer.finish();
  return DUGMA_OK;
}

// ---------------------------------------------------------------------------
// Scratch of dugma_energy_grad_noalloc: the pair kernel's per-workgroup
// partials (kPosePart doubles each) in a file-scope device array instead of
// the context's grow-only buffer.  Each GPU holds its own copy until the
// process ends; its address on a device comes from hipGetSymbolAddress with
// that device current (dugma_init calls noalloc_setup), and host code only
// ever passes that address.  Every partial record of a launch is written by
// its workgroup before k_reduce_parts reads it, so nothing is cleared.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocRecords = size_t(1) << 18;  // 16 MiB: 2^18 workgroups' partials
static __device__ __align__(256) double scratch[kNoAllocRecords * kPosePart];
constexpr int kNoAllocDevices = 64;
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[kNoAllocDevices];

int noalloc_setup(int device) {
  if (device < 0 || device >= kNoAllocDevices) return DUGMA_OK;  // the entry point reports it
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return DUGMA_OK;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
  g_scratch_ptr[device] = static_cast<double *>(p);
  return DUGMA_OK;
}

static double *noalloc_scratch(int device) {
  if (device < 0 || device >= kNoAllocDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[device];
}

}  // namespace dugma

using namespace dugma;

extern "C" int dugma_energy_grad_noalloc(dugma_ctx *ctx, const double *R, const double *t, int cov_mode,
                                         double *E, double *gpose) {
  int rc = check_pose_args(ctx, R, t);
  if (rc) return rc;
  double *sp = noalloc_scratch(ctx->device);
  if (!sp) return fail(DUGMA_ERR_STATE, "dugma_energy_grad_noalloc: no scratch address for this device");
  bool iso;
  rc = resolve_iso(ctx, cov_mode, &iso);
  if (rc) return rc;
  double res[kPosePart];
  rc = pose_pass(ctx, R, t, iso, kModePose, res, sp, kNoAllocRecords);
  if (rc) return rc;
  if (E) *E = res[0];
  const int nd = ctx->D == 3 ? 6 : 3;
  if (gpose)
    for (int a = 0; a < nd; ++a) gpose[a] = res[1 + a];
  return DUGMA_OK;
}

extern "C" int dugma_energy(dugma_ctx *ctx, const double *R, const double *t,
                            int cov_mode, double *E) {
  int rc = check_pose_args(ctx, R, t);
  if (rc) return rc;
  if (!E) return fail(DUGMA_ERR_ARG, "null E");
  bool iso;
  rc = resolve_iso(ctx, cov_mode, &iso);
  if (rc) return rc;
  double res[kPosePart];
  rc = pose_pass(ctx, R, t, iso, kModeEnergy, res);
  if (rc) return rc;
  *E = res[0];
  return DUGMA_OK;
}

extern "C" int dugma_energy_grad(dugma_ctx *ctx, const double *R,
                                 const double *t, int cov_mode, double *E,
                                 double *gpose) {
  int rc = check_pose_args(ctx, R, t);
  if (rc) return rc;
  bool iso;
  rc = resolve_iso(ctx, cov_mode, &iso);
  if (rc) return rc;
  double res[kPosePart];
  rc = pose_pass(ctx, R, t, iso, kModePose, res);
  if (rc) return rc;
  if (E) *E = res[0];
  const int nd = ctx->D == 3 ? 6 : 3;
  if (gpose)
    for (int a = 0; a < nd; ++a) gpose[a] = res[1 + a];
  return DUGMA_OK;
}

extern "C" int dugma_energy_grad_hess(dugma_ctx *ctx, const double *R, const double *t, int cov_mode, double *E,
                                      double *gpose, double *H) {
  int rc = check_pose_args(ctx, R, t);
  if (rc) return rc;
  if (ctx->D != 3) return fail(DUGMA_ERR_ARG, "dugma_energy_grad_hess: 3-D contexts only");
  bool iso;
  rc = resolve_iso(ctx, cov_mode, &iso);
  if (rc) return rc;
  double res[7], h[21];
  rc = pose_hess_pass(ctx, R, t, iso, res, h);
  if (rc) return rc;
  if (E) *E = res[0];
  if (gpose)
    for (int a = 0; a < 6; ++a) gpose[a] = res[1 + a];
  if (H) {
    int q = 0;
    for (int i = 0; i < 6; ++i)
      for (int j = i; j < 6; ++j, ++q) H[6 * i + j] = H[6 * j + i] = h[q];
  }
  return DUGMA_OK;
}

extern "C" int dugma_energy_grad_fd(dugma_ctx *ctx, const double *R,
                                    const double *t, int cov_mode, double h,
                                    double *E, double *gpose) {
  int rc = check_pose_args(ctx, R, t);
  if (rc) return rc;
  if (!(h > 0) || !std::isfinite(h)) return fail(DUGMA_ERR_ARG, "h must be positive");
  bool iso;
  rc = resolve_iso(ctx, cov_mode, &iso);
  if (rc) return rc;
  const int D = ctx->D, nd = D == 3 ? 6 : 3;
  double res[kPosePart];
  rc = pose_pass(ctx, R, t, iso, kModeEnergy, res);
  if (rc) return rc;
  if (E) *E = res[0];
  for (int k = 0; k < nd; ++k) {
    double p[6] = {0, 0, 0, 0, 0, 0}, Rn[9], tn[3], ep, em;
    p[k] = h;
    perturb(D, R, t, p, Rn, tn);
    rc = pose_pass(ctx, Rn, tn, iso, kModeEnergy, res);
    if (rc) return rc;
    ep = res[0];
    p[k] = -h;
    perturb(D, R, t, p, Rn, tn);
    rc = pose_pass(ctx, Rn, tn, iso, kModeEnergy, res);
    if (rc) return rc;
    em = res[0];
    if (gpose) gpose[k] = (ep - em) / (2.0 * h);
  }
  return DUGMA_OK;
}

extern "C" int dugma_energy_grad_points(dugma_ctx *ctx, const double *R,
                                        const double *t, int cov_mode,
                                        double *E, double *gpose, double *gX,
                                        double *gXC, double *gY, double *gYC,
                                        double *gdT) {
  int rc = check_pose_args(ctx, R, t);
  if (rc) return rc;
  if (cov_mode != DUGMA_COV_AUTO && cov_mode != DUGMA_COV_FULL && cov_mode != DUGMA_COV_ISO)
    return fail(DUGMA_ERR_ARG, "unknown cov_mode");
  dugma_ctx *c = ctx;
  const int D = c->D, DD = D * D, N = c->N, M = c->M;
  const int nacc = D == 3 ? kAcc3F : kAcc2F;
  const int nd = D == 3 ? 6 : 3;
  // Points left out of the records (non-finite) keep zero gradients.
  auto clear_points = [&]() {
    if (gX) std::fill(gX, gX + (size_t)N * D, 0.0);
    if (gXC) std::fill(gXC, gXC + (size_t)N * DD, 0.0);
    if (gY) std::fill(gY, gY + (size_t)M * D, 0.0);
    if (gYC) std::fill(gYC, gYC + (size_t)M * DD, 0.0);
  };
  if (gpose) std::fill(gpose, gpose + nd, 0.0);
  if (gdT) std::fill(gdT, gdT + (D == 3 ? 12 : 4), 0.0);
  if (E) *E = 0.0;
  if (c->nT == 0 || c->nS == 0) {
    clear_points();
    return DUGMA_OK;
  }

  // per-point passes use full-covariance records (isotropic points included)
  PoseArg ps = make_pose(c, R, t);
  const float lam_scale = pose_lam_scale(D, R);
  rc = transform_sources(c, ps, false, lam_scale);
  if (rc) return rc;
  const Sets onT = {0, c->dTrecF, c->dSrecF, lam_scale}, onS = {1, c->dSrecF, c->dTrecF, lam_scale};
  const size_t nT = c->nT, nS = c->nS;
  // Everything on the device is in scaled units: positions x s, covariances
  // x s^2, energy / s^D.
  const double cn = gauss_norm(D);
  const double sc = c->scale, sD = std::pow(sc, D);
  const double gpos = sD * sc;
  const PointUnits pu = {cn, gpos, sD * sc * sc};
  // device: the passes' sums | what goes to the host, targets | sources, each
  // workgroup sums, then the points' gradients, then the covariances'
  const size_t gridT = (nT + kBlock - 1) / kBlock, gridS = (nS + kBlock - 1) / kBlock;
  const size_t lenT = gridT * kPointSums + (size_t)N * (D + DD), lenS = gridS * kPointSums + (size_t)M * (D + DD);
  const size_t len_acc = (nT + nS) * nacc;
  rc = c->scratch2.ensure(sizeof(double) * (len_acc + lenT + lenS));
  if (rc) return rc;
  rc = c->hstage.ensure(sizeof(double) * (lenT + lenS));
  if (rc) return rc;
  double *acc = (double *)c->scratch2.ptr;
  double *dT = acc + len_acc, *dS = dT + lenT;
  double *hT = (double *)c->hstage.ptr, *hS = hT + lenT;
  if (!c->evpts) DUGMA_HIP(hipEventCreateWithFlags(&c->evpts, hipEventDisableTiming));
  // Target pass, its results on their way to the host, then the source pass:
  // the host hands the targets' gradients out while the source pass runs.
  // Points left out keep zero gradients.
  auto out = [&](bool tgt) -> int {
    const size_t n = tgt ? nT : nS, all = tgt ? N : M, grid = tgt ? gridT : gridS, len = tgt ? lenT : lenS;
    double *sums = tgt ? dT : dS, *P = sums + grid * kPointSums, *C = P + all * D;
    if (n < all) DUGMA_HIP(hipMemsetAsync(P, 0, sizeof(double) * all * (D + DD), c->stream));
    const double *a = tgt ? acc : acc + nT * nacc;
    const int *idx = tgt ? c->dTidx : c->dSidx;
#define POINTS_OUT(DD_, TT)                                                                                \
  hipLaunchKernelGGL((k_points_out<DD_, TT>), dim3((unsigned)grid), dim3(kBlock), 0, c->stream, a, c->dSsrc, idx, \
                     (int)n, ps, pu, P, C, sums)
    if (D == 3) {
      if (tgt) POINTS_OUT(3, true); else POINTS_OUT(3, false);
    } else {
      if (tgt) POINTS_OUT(2, true); else POINTS_OUT(2, false);
    }
#undef POINTS_OUT
    DUGMA_HIP(hipGetLastError());
    const bool points = tgt ? (gX || gXC) : (gY || gYC);
    DUGMA_HIP(hipMemcpyAsync(tgt ? hT : hS, sums, sizeof(double) * (points ? len : grid * kPointSums),
                             hipMemcpyDeviceToHost, c->stream));
    return DUGMA_OK;
  };
  rc = point_pass(c, onT, ps, 1, acc);
  if (!rc) rc = out(true);
  if (rc) return rc;
  hipError_t e = hipEventRecord(c->evpts, c->stream);
  if (e != hipSuccess) return hip_fail(e, "dugma_energy_grad_points: event");
  rc = point_pass(c, onS, ps, 2, acc + nT * nacc);
  if (!rc) rc = out(false);
  if (rc) return rc;
  // the caller's arrays, in pieces, on a few threads (fresh pages are touched
  // here for the first time: a serial fill of them took 2 ms)
  auto hand_out = [&](const double *P, size_t all, double *gP, double *gC) {
    const size_t np = gP ? all * D : 0, nc = gC ? all * DD : 0;
    const double *C = P + all * D;
    constexpr size_t kPiece = size_t(1) << 16;  // 512 KiB
    const size_t kp = (np + kPiece - 1) / kPiece, kc = (nc + kPiece - 1) / kPiece;
    parallel_for(kp + kc, [&](size_t q) {
      const size_t o = (q < kp ? q : q - kp) * kPiece;
      if (q < kp)
        memcpy(gP + o, P + o, sizeof(double) * std::min(kPiece, np - o));
      else
        memcpy(gC + o, C + o, sizeof(double) * std::min(kPiece, nc - o));
    });
  };
  e = hipEventSynchronize(c->evpts);
  if (e != hipSuccess) return hip_fail(e, "dugma_energy_grad_points: download");
  hand_out(hT + gridT * kPointSums, N, gX, gXC);
  e = hipStreamSynchronize(c->stream);  // the source pass and its results
  if (e != hipSuccess) return hip_fail(e, "dugma_energy_grad_points: download");
  hand_out(hS + gridS * kPointSums, M, gY, gYC);
  double Etot = 0.0, ps_sum[kPointSums] = {0.0};
  for (size_t q = 0; q < gridT; ++q) Etot += hT[q * kPointSums];
  for (size_t q = 0; q < gridS; ++q)
    for (int a = 1; a < kPointSums; ++a) ps_sum[a] += hS[q * kPointSums + a];
  if (E) *E = cn * Etot * sD;
  const double *gw = ps_sum + 1, gth = ps_sum[1], *gt = ps_sum + 4, *G = ps_sum + 7;
  // unscale: rotation / dR parts ~ s^D, translation parts ~ s^(D+1)
  if (gpose) {
    if (D == 3) {
      for (int a = 0; a < 3; ++a) {
        gpose[a] = gw[a] * sD;
        gpose[3 + a] = gt[a] * gpos;
      }
    } else {
      gpose[0] = gth * sD;
      gpose[1] = gt[0] * gpos;
      gpose[2] = gt[1] * gpos;
    }
  }
  if (gdT) {
    if (D == 3) {
      // energy3D.m variable order: t1 t2 t3 r11 r12 r13 r21 ... r33 (dR row-major)
      for (int a = 0; a < 3; ++a) gdT[a] = gt[a] * gpos;
      for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) gdT[3 + 3 * a + b] = G[a + 3 * b] * sD;
    } else {
      // energy2D.m: t1 t2 r11 r21 with dR = [[r11, -r21], [r21, r11]]
      gdT[0] = gt[0] * gpos;
      gdT[1] = gt[1] * gpos;
      gdT[2] = (G[0] + G[3]) * sD;
      gdT[3] = (G[1] - G[2]) * sD;
    }
  }
  return DUGMA_OK;
}

extern "C" int dugma_autotune(dugma_ctx *ctx, int cov_mode) {
  if (!ctx) return fail(DUGMA_ERR_ARG, "dugma_autotune: null context");
  bool iso;
  int rc = resolve_iso(ctx, cov_mode, &iso);
  if (rc) return rc;
  if (ctx->nT == 0 || ctx->nS == 0) return DUGMA_OK;
  const int D = ctx->D;
  double R[9] = {0}, t[3] = {0, 0, 0};
  for (int a = 0; a < D; ++a) R[a * (D + 1)] = 1.0;
  hipEvent_t e0, e1;
  DUGMA_HIP(hipEventCreate(&e0));
  DUGMA_HIP(hipEventCreate(&e1));
  static const int kW[] = {2048, 4096, 8192, 16384, 32768};
  const double pairs = (double)ctx->nT * ctx->nS;
  const int reps = pairs > 4e9 ? 1 : (pairs > 1e8 ? 3 : 10);
  for (int m = 0; m < 2; ++m) {
    const int mode = m == 0 ? kModeEnergy : kModePose;
    dugma_ctx::Tuned best;
    float best_ms = 1e30f;
    // the stationary and streamed sets of pose_pass
    const int nP = sources_stationary() ? ctx->nS : ctx->nT, nQ = sources_stationary() ? ctx->nT : ctx->nS;
    int last_split = -1;
    for (const int waves : kW) {
      dugma_ctx::Tuned &tu = ctx->tuned[m][iso ? 1 : 0];
      tu.T = 1;
      tu.target_waves = waves;
      // targets that give the launch of the previous one are not timed again
      const int split = ctx_plan(ctx, nP, nQ, mode, iso).qsplit;
      if (split == last_split) continue;
      last_split = split;
      double res[kPosePart];
      rc = pose_pass(ctx, R, t, iso, mode, res);  // warm
      if (rc) break;
      (void)hipEventRecord(e0, ctx->stream);
      for (int r = 0; r < reps && !rc; ++r) rc = pose_pass(ctx, R, t, iso, mode, res);
      (void)hipEventRecord(e1, ctx->stream);
      (void)hipEventSynchronize(e1);
      float ms = 0.0f;
      (void)hipEventElapsedTime(&ms, e0, e1);
      if (!rc && ms < best_ms) {
        best_ms = ms;
        best = tu;
      }
    }
    ctx->tuned[m][iso ? 1 : 0] = best;
    if (rc) break;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

extern "C" int dugma_ctx_plan(const dugma_ctx *ctx, int cov_mode, int *lane_points,
                              int *target_waves) {
  if (!ctx) return fail(DUGMA_ERR_ARG, "dugma_ctx_plan: null context");
  const bool iso = cov_mode == DUGMA_COV_ISO || (cov_mode == DUGMA_COV_AUTO && ctx->iso);
  const dugma_ctx::Tuned &tu = ctx->tuned[1][iso ? 1 : 0];
  if (lane_points) *lane_points = tu.T;
  if (target_waves) *target_waves = tu.target_waves;
  return DUGMA_OK;
}
