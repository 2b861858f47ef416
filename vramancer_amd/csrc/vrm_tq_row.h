// One row of the TurboQuant encoder on one wavefront, operation by operation
// as the reference evaluates it (IEEE binary32, the C library's atan2): the
// path every code is defined by.  The row lives in LDS between stages.
#pragma once
#include "vrm_common.h"
#include "vrm_fdlibm_atan2f.h"
#include "vrm_tq_common.h"

#include <math.h>

namespace vrm {
namespace {

#pragma clang fp contract(off)

// Element e of the polar decode of one row from the fp32 radius and the
// level-major bins (level l at offset PD - (PD >> l)).  The reference decodes
// level by level from the top, each value r of level l becoming the pair
// (r cos, r sin) of level l - 1; element e is therefore the product chain
//   ((radius * f_{NL-1}) * f_{NL-2}) ... * f_0,
// f_l the cos (bit l of e clear) or sin (set) of angle e >> (l + 1) of level
// l, the same roundings in the same order, with no exchange between lanes.
template <int PD>
__device__ __forceinline__ float polar_element(float radius, const uint8_t* bins, const float* lut, int nb, int e) {
  constexpr int NL = __builtin_ctz(PD);
  float r = radius;
#pragma unroll
  for (int l = NL - 1; l >= 0; --l) {
    const int idx = min((int)bins[PD - (PD >> l) + (e >> (l + 1))], nb - 1);  // caller-supplied bins stay in the table
    r = __fmul_rn(r, lut[(l == 0 ? 0 : 2 * nb) + (((e >> l) & 1) ? nb : 0) + idx]);
  }
  return r;
}

// Polar decode of one row into `recon` (LDS, PD floats); bins may have been
// written by any lane before the call, recon is visible to every lane after.
template <int PD>
__device__ __forceinline__ void polar_decode(float radius, const uint8_t* bins, const float* lut, int nb,
                                             float* recon, int lane) {
  row_sync();
#pragma unroll
  for (int k = 0; k < tq_per_lane(PD); ++k)
    if (k * 64 + lane < PD) recon[k * 64 + lane] = polar_element<PD>(radius, bins, lut, nb, k * 64 + lane);
  row_sync();
}

// LDS working set of one row.
template <int PD>
struct RowLds {
  float rot[PD];               // rotated row
  float rad[PD];               // radius of each polar node, level-major like the bins
  alignas(16) double res[PD];  // QJL residual, widened once by the lane that owns it
  uint8_t bins[PD];
  float norm_acc[8];
};

// Rotation and polar encoding of one row (source element e is load(e) for
// e < head_dim, zero padding above): leaves the level-major bins in w.bins,
// the rotated row in v (element e in lane e % 64, register e / 64; lanes past
// a row of fewer than 64 elements hold zeros) and in w.rot, and returns the
// fp32 final radius.
template <int PD, typename Load>
__device__ __forceinline__ float encode_row(Load load, int head_dim, const float* signs, int bits,
                                            float (&v)[tq_per_lane(PD)], RowLds<PD>& w, int lane) {
  constexpr int PER = tq_per_lane(PD);
  constexpr int NL = __builtin_ctz(PD);
  const int nb = 1 << bits;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = k * 64 + lane;
    const float x = e < head_dim ? load(e) : 0.f;
    v[k] = e < PD ? __fmul_rn(x, signs[e]) : 0.f;
  }
  fwht<PD>(v, lane);
  const float root = (float)sqrt((double)PD);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    v[k] = __fdiv_rn(v[k], root);
    if (k * 64 + lane < PD) w.rot[k * 64 + lane] = v[k];
  }
  row_sync();

  // The radii only need square roots, level after level: node i of level l
  // (w.rad[PD - (PD >> l) + i]) over children 2 i, 2 i + 1 of level l - 1
  // (the rotated row below level 0).
  for (int level = 0; level < NL; ++level) {
    const float* child = level == 0 ? w.rot : w.rad + (PD - (PD >> (level - 1)));
    float* rad = w.rad + (PD - (PD >> level));
    for (int i = lane; i < (PD >> (level + 1)); i += 64) {
      const float x0 = child[2 * i], x1 = child[2 * i + 1];
      rad[i] = sqrt_rn(__fadd_rn(__fadd_rn(__fmul_rn(x0, x0), __fmul_rn(x1, x1)), 1e-12f));
    }
    row_sync();
  }
  // With every child known, the angles of all levels are independent: lane
  // takes bins b = lane, lane + 64, ... of the level-major order.
  const float lo0 = (float)-3.141592653589793, range0 = (float)6.283185307179586;
  const float range1 = (float)1.5707963267948966;
  const float nbf = (float)nb;
  for (int b = lane; b < PD - 1; b += 64) {
    const int level = NL - 1 - (31 - __builtin_clz(PD - b - 1));  // PD >> (level + 1) < PD - b <= PD >> level
    const int i = b - (PD - (PD >> level));
    const float* child = level == 0 ? w.rot : w.rad + (PD - (PD >> (level - 1)));
    const float x0 = child[2 * i], x1 = child[2 * i + 1];
    const float th = vrm_fdlibm::atan2f(x1, x0);
    const float nrm = level == 0 ? __fdiv_rn(__fsub_rn(th, lo0), range0) : __fdiv_rn(th, range1);
    int idx = (int)__fmul_rn(nrm, nbf);  // truncation toward zero, as .long()
    idx = min(max(idx, 0), nb - 1);
    w.bins[b] = (uint8_t)idx;
  }
  row_sync();
  return w.rad[PD - 2];
}

// Residual against the reconstruction from the fp32 radius, its QJL signs
// (float64 dot products; sign(j) is handed to put_sign) and the residual norm
// as PyTorch's CPU 2-norm reduces a row: eight interleaved fused accumulators
// summed in order for rows of 4 floats or more, one fused chain for a row of
// 2 (measured against torch.norm at 2 .. 256 floats).  Returns the norm.
template <int PD, typename PutSign>
__device__ __forceinline__ float qjl_row(const float (&v)[tq_per_lane(PD)], float radius, const float* lut, int bits,
                                         const float* jl, int qjl_dim, RowLds<PD>& w, int lane, PutSign put_sign) {
  constexpr int PER = tq_per_lane(PD);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = k * 64 + lane;
    if (e < PD) w.res[e] = (double)__fsub_rn(v[k], polar_element<PD>(radius, w.bins, lut, 1 << bits, e));
  }
  row_sync();
  // Lane j walks row j of the JL matrix.  With a 16-byte aligned matrix (every
  // row is then aligned, PD being a multiple of 4) it reads four floats per
  // load; the residual comes as doubles, two per LDS broadcast.  The
  // accumulation order is the element order either way.
  const bool vec = PD >= 4 && (reinterpret_cast<uintptr_t>(jl) & 15) == 0;
  const double2* r2 = reinterpret_cast<const double2*>(w.res);
  for (int j = lane; j < qjl_dim; j += 64) {
    const float* jr = jl + (size_t)j * PD;
    double s = 0.0;
    if (vec) {
      const float4* jr4 = reinterpret_cast<const float4*>(jr);
#pragma unroll 8
      for (int m = 0; m < PD / 4; ++m) {
        const float4 x = jr4[m];
        const double2 ra = r2[2 * m], rb = r2[2 * m + 1];
        s = fma(ra.x, (double)x.x, s);
        s = fma(ra.y, (double)x.y, s);
        s = fma(rb.x, (double)x.z, s);
        s = fma(rb.y, (double)x.w, s);
      }
    } else {
      for (int e = 0; e < PD; ++e) s = fma(w.res[e], (double)jr[e], s);
    }
    put_sign(j, s > 0.0);
  }
  if constexpr (PD == 2) {
    const float x0 = (float)w.res[0], x1 = (float)w.res[1];  // exact: widened from floats
    return sqrt_rn(fmaf(x1, x1, __fmul_rn(x0, x0)));
  }
  if (lane < 8) {
    float acc = 0.f;
#pragma unroll
    for (int m = 0; m < (PD + 7) / 8; ++m) {
      if (lane + 8 * m < PD) {
        const float x = (float)w.res[lane + 8 * m];  // exact: widened from a float
        acc = fmaf(x, x, acc);
      }
    }
    w.norm_acc[lane] = acc;
  }
  row_sync();
  float s = w.norm_acc[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) s = __fadd_rn(s, w.norm_acc[k]);
  return sqrt_rn(s);
}

}  // namespace
}  // namespace vrm
