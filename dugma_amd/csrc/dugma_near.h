// dugma_near.h -- spatial index of the two clouds, shared by the kernels that
// leave out pairs whose term is exactly zero.
//
// A pair's term is e = exp2(x) det(S)^-1/2 with x = -log2(e)/2 d^T S^-1 d, and
// v_exp_f32 returns exactly 0 for x < -126 (denormal results are flushed):
// such a pair adds +0 to every FP32 sum, so leaving it out changes no bit.
// d^T S^-1 d >= |d|^2 / (lam_p + lam_q), lam the largest eigenvalue of each
// point's covariance, so every pair with |d|^2 > kZeroDist2 (lam_p + lam_q) is
// such a pair.  kZeroDist2 = 126 * 2 ln 2 plus 1% for the rounding of the FP32
// exponent; lam itself is raised where a covariance's conditioning makes that
// rounding larger.
//
// Each cloud's kept points are put once, at init, into the order of a Hilbert
// curve; 64 consecutive ones are a block with a bounding box and the largest
// lam of its points.  The order only says which points share a wave or a box:
// the sums over the streamed points keep their own order and grouping.
#pragma once

#include "dugma_internal.h"

namespace dugma {

constexpr float kZeroDist2 = 176.42f;

// 64 consecutive points in Hilbert order: bounding box, largest lam.
struct alignas(16) QBox {
  float lo[3], lam;
  float hi[3], pad;
};

// A point in Hilbert order: position (hi part) and lam.
struct alignas(16) QAux {
  float x, y, z, lam;
};

// True unless every pair of a point (or box) in [lx, hx] x ... with lam and a
// point of box b is certain to have an exactly zero term.  A gap that is not
// finite counts as near (the dense sums would carry the infinity or NaN on).
__device__ __forceinline__ bool box_near(const QBox &b, float lx, float ly, float lz, float hx, float hy,
                                         float hz, float lam) {
  const float gx = fmaxf(fmaxf(b.lo[0] - hx, lx - b.hi[0]), 0.0f);
  const float gy = fmaxf(fmaxf(b.lo[1] - hy, ly - b.hi[1]), 0.0f);
  const float gz = fmaxf(fmaxf(b.lo[2] - hz, lz - b.hi[2]), 0.0f);
  const float g2 = fmaf(gx, gx, fmaf(gy, gy, gz * gz));
  return !(g2 > kZeroDist2 * (b.lam + lam) && g2 < __builtin_huge_valf());
}

// Minimum / maximum over each row of 16 lanes, in every lane of the row.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float row_min(float v) {
  v = fminf(v, dpp_f<0x128>(v));
  v = fminf(v, dpp_f<0x124>(v));
  v = fminf(v, dpp_f<0x122>(v));
  return fminf(v, dpp_f<0x121>(v));
}
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, dpp_f<0x128>(v));
  v = fmaxf(v, dpp_f<0x124>(v));
  v = fmaxf(v, dpp_f<0x122>(v));
  return fmaxf(v, dpp_f<0x121>(v));
}

// Minimum / maximum over each 4 lanes, in every one of them (DPP quad_perm).
__device__ __forceinline__ float quad_min(float v) {
  v = fminf(v, dpp_f<0xB1>(v));     // [1, 0, 3, 2]
  return fminf(v, dpp_f<0x4E>(v));  // [2, 3, 0, 1]
}
__device__ __forceinline__ float quad_max(float v) {
  v = fmaxf(v, dpp_f<0xB1>(v));
  return fmaxf(v, dpp_f<0x4E>(v));
}

// The index's arrays: their size, and where they lie.
size_t near_bytes(int nT, int nS);
void near_place(dugma_ctx *c, char *base);
// Hilbert order of both clouds (init): lo, hi are the kept points' bounds.
int near_build(dugma_ctx *c, const double lo[2][3], const double hi[2][3]);
// lam, aux and boxes again after covariances changed on the device; cloud 0
// targets, 1 sources.
int near_refresh(dugma_ctx *c, int cloud);
// aux and boxes of the transformed sources (recs: this call's source records
// in kept order; lam times lam_scale).
int near_index_sources(dugma_ctx *c, bool iso, const void *recs, float lam_scale);

}  // namespace dugma
