// dugma_near.hip -- Hilbert order and bounding boxes of the two clouds
// (dugma_near.h says what they are for).
#include <algorithm>
#include <cmath>

#include <hipcub/hipcub.hpp>

#include "dugma_internal.h"
#include "dugma_near.h"
#include "dugma_pairs.h"

namespace dugma {

constexpr int kNBlock = 256;

struct KeyBox {
  float lo[3], inv[3];  // lower corner; cells per unit length
};

// Position along a Hilbert curve of a cell with D coordinates of B bits each
// (J. Skilling, "Programming the Hilbert curve", 2004: the coordinates to the
// transposed index, whose bits are then interleaved).  Consecutive positions are
// neighbouring cells, so 64 points in a row seldom straddle distant parts of
// the cloud: at 6,000 structured-light points with outliers a workgroup's boxes
// reach 160 streamed points, with a Morton order 240 (the largest 430 and 1,150).
template <int D, int B>
__device__ __forceinline__ unsigned hilbert_key(unsigned *x) {
  for (unsigned q = 1u << (B - 1); q > 1; q >>= 1) {
    const unsigned m = q - 1;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      if (x[a] & q) {
        x[0] ^= m;
      } else {
        const unsigned t = (x[0] ^ x[a]) & m;
        x[0] ^= t;
        x[a] ^= t;
      }
    }
  }
#pragma unroll
  for (int a = 1; a < D; ++a) x[a] ^= x[a - 1];
  unsigned t = 0;
  for (unsigned q = 1u << (B - 1); q > 1; q >>= 1)
    if (x[D - 1] & q) t ^= q - 1;
  unsigned k = 0;
  for (int b = B - 1; b >= 0; --b)
#pragma unroll
    for (int a = 0; a < D; ++a) k = (k << 1) | (((x[a] ^ t) >> b) & 1u);
  return k;
}

// 30-bit Hilbert key of kept point q (init's FP32 point of index idx[q]).
template <int D>
__global__ __launch_bounds__(kNBlock) void k_near_keys(const float *__restrict__ P, const int *__restrict__ idx,
                                                       int n, KeyBox kb, unsigned *__restrict__ key,
                                                       int *__restrict__ val) {
  constexpr int B = D == 3 ? 10 : 15;
  const int q = blockIdx.x * kNBlock + threadIdx.x;
  if (q >= n) return;
  const float *p = P + (size_t)idx[q] * D;
  unsigned x[D];
#pragma unroll
  for (int a = 0; a < D; ++a)
    x[a] = (unsigned)fminf(fmaxf((p[a] - kb.lo[a]) * kb.inv[a], 0.0f), (float)((1 << B) - 1));  // NaN -> 0
  key[q] = hilbert_key<D, B>(x);
  val[q] = q;
}

// How much a covariance's conditioning loosens the bound: the FP32 determinant
// of a pair's S is off by up to 1e-6 of its mean eigenvalue cubed (in 2-D
// squared), so d^T S^-1 d by that share of 1 / dn, dn the determinant over that
// cube; by Minkowski's inequality a pair is no worse than three times its worse
// point.  Near 1e-6 the FP32 determinant can come out as 0 or negative and the
// term as a NaN: such a point counts as near everything.
__device__ __forceinline__ float lam_slack(float dn) {
  return dn > 4e-6f ? 1.001f + 6e-6f / dn : __builtin_huge_valf();
}
// Largest eigenvalue of a symmetric covariance (closed form, FP32), raised by
// 1e-3 and by lam_slack so that it is a bound.
__device__ __forceinline__ float lam_max3(float s11, float s12, float s13, float s22, float s23, float s33) {
  const float m = (s11 + s22 + s33) * (1.0f / 3.0f);
  const float d1 = s11 - m, d2 = s22 - m, d3 = s33 - m;
  const float o2 = s12 * s12 + s13 * s13 + s23 * s23;
  const float p = sqrtf((d1 * d1 + d2 * d2 + d3 * d3 + 2.0f * o2) * (1.0f / 6.0f));
  if (!(p > 1e-6f * m)) return m * 1.001f + 2.0f * p;  // s I (or NaN)
  const float im = 1.0f / m;
  const float n11 = s11 * im, n22 = s22 * im, n33 = s33 * im, n12 = s12 * im, n13 = s13 * im, n23 = s23 * im;
  const float dn = n11 * (n22 * n33 - n23 * n23) - n12 * (n12 * n33 - n23 * n13) + n13 * (n12 * n23 - n22 * n13);
  const float ip = 1.0f / p;
  const float b11 = d1 * ip, b22 = d2 * ip, b33 = d3 * ip, b12 = s12 * ip, b13 = s13 * ip, b23 = s23 * ip;
  const float det = b11 * (b22 * b33 - b23 * b23) - b12 * (b12 * b33 - b23 * b13) + b13 * (b12 * b23 - b22 * b13);
  const float r = fminf(1.0f, fmaxf(-1.0f, 0.5f * det));
  return (m + 2.0f * p * cosf(acosf(r) * (1.0f / 3.0f))) * lam_slack(dn);
}
__device__ __forceinline__ float rec_lam(const Rec3F &r) {
  return lam_max3(r.s11, r.s12, r.s13, r.s22, r.s23, r.s33);
}
__device__ __forceinline__ float rec_lam(const Rec2F &r) {
  const float h = 0.5f * (r.s11 + r.s22), d = 0.5f * (r.s11 - r.s22);
  const float ih = 1.0f / h;
  const float dn = (r.s11 * ih) * (r.s22 * ih) - (r.s12 * ih) * (r.s12 * ih);
  return (h + sqrtf(d * d + r.s12 * r.s12)) * lam_slack(dn);
}
__device__ __forceinline__ void rec_pos(const Rec3F &r, float *x) { x[0] = r.hx; x[1] = r.hy; x[2] = r.hz; }
__device__ __forceinline__ void rec_pos(const Rec3I &r, float *x) { x[0] = r.hx; x[1] = r.hy; x[2] = r.hz; }
__device__ __forceinline__ void rec_pos(const Rec2F &r, float *x) { x[0] = r.hx; x[1] = r.hy; x[2] = 0.0f; }
__device__ __forceinline__ void rec_pos(const Rec2I &r, float *x) { x[0] = r.hx; x[1] = r.hy; x[2] = 0.0f; }

// aux and box of one 64-point block, one wave each: lanes past n hold the last
// point.
__device__ __forceinline__ void write_block(const float *x, float lam, int pos, int n, QAux *__restrict__ aux,
                                            QBox *__restrict__ box) {
  if (pos < n) {
    QAux a;
    a.x = x[0];
    a.y = x[1];
    a.z = x[2];
    a.lam = lam;
    aux[pos] = a;
  }
  float v[7] = {x[0], x[1], x[2], x[0], x[1], x[2], lam};
#pragma unroll
  for (int a = 0; a < 7; ++a) {
    v[a] = a < 3 ? row_min(v[a]) : row_max(v[a]);
#pragma unroll
    for (int m = 16; m < 64; m <<= 1) {
      const float o = __shfl_xor(v[a], m, 64);
      v[a] = a < 3 ? fminf(v[a], o) : fmaxf(v[a], o);
    }
  }
  if ((threadIdx.x & 63) == 0) {
    QBox b;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      // wide enough for the positions' lo parts
      const float slack = 2.4e-7f * fmaxf(fabsf(v[a]), fabsf(v[3 + a]));
      b.lo[a] = v[a] - slack;
      b.hi[a] = v[3 + a] + slack;
    }
    b.lam = v[6];
    b.pad = 0.0f;
    box[pos >> 6] = b;
  }
}

// The cloud's own index: lam from the full records.
template <class Rec>
__global__ __launch_bounds__(kNBlock) void k_near_index(const Rec *__restrict__ recs, const int *__restrict__ ord,
                                                        int n, float *__restrict__ lam, QAux *__restrict__ aux,
                                                        QBox *__restrict__ box) {
  const int pos = blockIdx.x * kNBlock + threadIdx.x;
  if ((pos & ~63) >= n) return;  // whole wave
  const Rec r = recs[ord[min(pos, n - 1)]];
  float x[3];
  rec_pos(r, x);
  const float l = rec_lam(r);
  if (pos < n) lam[pos] = l;
  write_block(x, l, pos, n, aux, box);
}

// The sources' lam from the FP64 source data (their records are per call).
template <int D>
__global__ __launch_bounds__(kNBlock) void k_near_lam_src(const double *__restrict__ src,
                                                          const int *__restrict__ ord, int n,
                                                          float *__restrict__ lam) {
  const int pos = blockIdx.x * kNBlock + threadIdx.x;
  if (pos >= n) return;
  const double *S = src + (size_t)ord[pos] * (D + D * D) + D;
  if (D == 3) {
    lam[pos] = lam_max3((float)S[0], (float)S[3], (float)S[6], (float)S[4], (float)S[7], (float)S[8]);
  } else {
    Rec2F r;
    r.s11 = (float)S[0];
    r.s12 = (float)S[2];
    r.s22 = (float)S[3];
    lam[pos] = rec_lam(r);
  }
}

// This call's transformed sources: lam kept from the index.
template <class Rec>
__global__ __launch_bounds__(kNBlock) void k_near_index_src(const Rec *__restrict__ recs,
                                                            const int *__restrict__ ord, int n,
                                                            const float *__restrict__ lam, float lam_scale,
                                                            QAux *__restrict__ aux, QBox *__restrict__ box) {
  const int pos = blockIdx.x * kNBlock + threadIdx.x;
  if ((pos & ~63) >= n) return;  // whole wave
  const int q = min(pos, n - 1);
  const Rec r = recs[ord[q]];
  float x[3];
  rec_pos(r, x);
  write_block(x, lam[q] * lam_scale, pos, n, aux, box);
}

static dim3 near_grid(int n) { return dim3((unsigned)((n + kNBlock - 1) / kNBlock)); }

int near_refresh(dugma_ctx *c, int cloud) {
  NearCloud &nc = c->near[cloud];
  const int n = cloud == 0 ? c->nT : c->nS;
  if (n == 0) return DUGMA_OK;
  const dim3 blk(kNBlock);
  if (cloud == 0) {
    if (c->D == 3)
      hipLaunchKernelGGL(k_near_index<Rec3F>, near_grid(n), blk, 0, c->stream, (const Rec3F *)c->dTrecF, nc.ord, n,
                         nc.lam, nc.aux, nc.box);
    else
      hipLaunchKernelGGL(k_near_index<Rec2F>, near_grid(n), blk, 0, c->stream, (const Rec2F *)c->dTrecF, nc.ord, n,
                         nc.lam, nc.aux, nc.box);
  } else {
    if (c->D == 3)
      hipLaunchKernelGGL(k_near_lam_src<3>, near_grid(n), blk, 0, c->stream, c->dSsrc, nc.ord, n, nc.lam);
    else
      hipLaunchKernelGGL(k_near_lam_src<2>, near_grid(n), blk, 0, c->stream, c->dSsrc, nc.ord, n, nc.lam);
  }
  DUGMA_HIP(hipGetLastError());
  return DUGMA_OK;
}

int near_index_sources(dugma_ctx *c, bool iso, const void *recs, float lam_scale) {
  NearCloud &nc = c->near[1];
  const int n = c->nS;
  const dim3 blk(kNBlock);
#define NEAR_SRC(R)                                                                                             \
  hipLaunchKernelGGL(k_near_index_src<R>, near_grid(n), blk, 0, c->stream, (const R *)recs, nc.ord, n, nc.lam, \
                     lam_scale, nc.aux, nc.box)
  if (c->D == 3) {
    if (iso) NEAR_SRC(Rec3I); else NEAR_SRC(Rec3F);
  } else {
    if (iso) NEAR_SRC(Rec2I); else NEAR_SRC(Rec2F);
  }
#undef NEAR_SRC
  DUGMA_HIP(hipGetLastError());
  return DUGMA_OK;
}

static size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

size_t near_bytes(int nT, int nS) {
  size_t bytes = 0;
  for (const size_t m : {(size_t)nT, (size_t)nS})
    bytes += al256(m * sizeof(int)) + al256(m * sizeof(QAux)) + al256((m + 63) / 64 * sizeof(QBox)) +
             al256(m * sizeof(float));
  return bytes;
}

void near_place(dugma_ctx *c, char *b) {
  for (int w = 0; w < 2; ++w) {
    NearCloud &nc = c->near[w];
    const size_t m = w == 0 ? c->nT : c->nS;
    nc.ord = (int *)b;
    b += al256(m * sizeof(int));
    nc.aux = (QAux *)b;
    b += al256(m * sizeof(QAux));
    nc.box = (QBox *)b;
    b += al256((m + 63) / 64 * sizeof(QBox));
    nc.lam = (float *)b;
    b += al256(m * sizeof(float));
  }
}

int near_build(dugma_ctx *c, const double lo[2][3], const double hi[2][3]) {
  const int n[2] = {c->nT, c->nS};
  const int nmax = std::max(n[0], n[1]);
  if (nmax == 0) return DUGMA_OK;
  size_t tmp = 0;
  DUGMA_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, (const unsigned *)nullptr, (unsigned *)nullptr,
                                               (const int *)nullptr, (int *)nullptr, nmax, 0, 30, c->stream));
  const size_t bk = al256((size_t)nmax * 4);
  // not the context's scratch: growing that in the first call would cost it a
  // free (55 us)
  struct Temp : DevBuf {
    ~Temp() { release(); }
  } temp;
  int rc = temp.ensure(3 * bk + tmp);
  if (rc) return rc;
  char *sb = (char *)temp.ptr;
  unsigned *k0 = (unsigned *)sb, *k1 = (unsigned *)(sb + bk);
  int *v0 = (int *)(sb + 2 * bk);
  void *st = sb + 3 * bk;
  const int D = c->D;
  for (int w = 0; w < 2; ++w) {
    NearCloud &nc = c->near[w];
    if (n[w] == 0) continue;
    // cubic cells over the largest extent
    double ext = 0.0;
    for (int a = 0; a < D; ++a) ext = std::max(ext, hi[w][a] - lo[w][a]);
    KeyBox kb;
    const double cells = D == 3 ? 1023.0 : 32767.0;
    const double inv = ext > 0.0 && std::isfinite(cells / ext) ? cells / ext : 0.0;
    for (int a = 0; a < 3; ++a) {
      kb.lo[a] = a < D ? (float)lo[w][a] : 0.0f;
      kb.inv[a] = a < D ? (float)inv : 0.0f;
    }
    const float *P = w == 0 ? c->dX : c->dY;
    const int *idx = w == 0 ? c->dTidx : c->dSidx;
    if (D == 3)
      hipLaunchKernelGGL(k_near_keys<3>, near_grid(n[w]), dim3(kNBlock), 0, c->stream, P, idx, n[w], kb, k0, v0);
    else
      hipLaunchKernelGGL(k_near_keys<2>, near_grid(n[w]), dim3(kNBlock), 0, c->stream, P, idx, n[w], kb, k0, v0);
    DUGMA_HIP(hipGetLastError());
    DUGMA_HIP(hipcub::DeviceRadixSort::SortPairs(st, tmp, k0, k1, v0, nc.ord, n[w], 0, 30, c->stream));
    rc = near_refresh(c, w);
    if (rc) return rc;
  }
  DUGMA_HIP(hipStreamSynchronize(c->stream));  // the sort's memory goes
  return DUGMA_OK;
}

}  // namespace dugma
