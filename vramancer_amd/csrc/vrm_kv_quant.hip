// Quantize-on-append for the int8 and fp8-e4m3 paged pools, bulk page writes
// (prefill) and page dequantization.
//
// The reference writes raw K/V rows with an index-put
// (core/paged_attention.py:611-612, pool[page, layer, 0|1, :, slot, :] = k|v)
// and has no int8/fp8 codec; the codecs here are this library's definitions:
//   int8: per (token, head) scale = amax / 127, code = clamp(rne(x / scale), +-127)
//   fp8 : per (page, head) scale = amax / 448, code = e4m3fn_rne(x / scale)
// Divisions are IEEE round-to-nearest so codes are bit-identical to the same
// formulas evaluated with PyTorch on the CPU.
//
// Layout of a quantized (page, layer, K/V, head) slice of PS x D codes: K is
// token-major (code of token t, dim d at t * D + d, as the reference's pool);
// V is tiled, code of token t, dim d at
//   ((t / 4 * 16 + d % 16) * (D / 16) + d / 16) * 4 + t % 4,
// so that a decode lane finds the 4 tokens of its MFMA k-slice for the dims
// col, col + 16, ... of its operand row in D / 4 consecutive bytes.
#include "vrm_common.h"

#include <math.h>

namespace vrm {
namespace {

bool quant_pool(int kv_dtype) {
  return kv_dtype == VRM_KV_I8 || kv_dtype == VRM_KV_FP8E4M3 || inline_pool(kv_dtype);
}
bool fp8_pool(int kv_dtype) { return kv_dtype == VRM_KV_FP8E4M3 || kv_dtype == VRM_KV_FP8E4M3_INLINE; }


template <int SRC>
__device__ __forceinline__ float load_src(const void* p, size_t i) {
  if constexpr (SRC == VRM_SRC_F32) {
    return static_cast<const float*>(p)[i];
  } else if constexpr (SRC == VRM_SRC_F16) {
    return f16_bits_to_f32(static_cast<const uint16_t*>(p)[i]);
  } else {
    return bf16_bits_to_f32(static_cast<const uint16_t*>(p)[i]);
  }
}

__device__ __forceinline__ int8_t int8_code(float x, float scale) {
  if (!(scale > 0.f)) return 0;
  float r = rintf(__fdiv_rn(x, scale));
  r = fminf(fmaxf(r, -127.f), 127.f);
  return (int8_t)(int)r;
}

__device__ __forceinline__ uint8_t fp8_code(float x, float scale) {
  if (!(scale > 0.f)) return 0;
  return vrm_e4m3::encode(__fdiv_rn(x, scale));
}

struct QuantArgs {
  const void* key;
  const void* value;
  const int32_t* page_ids;
  const int32_t* slots;    // append: slot of each token; pages: valid tokens per page
  uint8_t* pool;
  float* scales;
  int KH, L, P, layer;
  int D, PS;               // head_dim (multiple of 16, <= 256) and page size (multiple of 4)
  PoolGeom g;              // plain or inline layout of codes and scales
};

// Codes of the (page, layer, K/V, kv-head) slice and its scales (int8: PS of
// them, one per token; fp8: one).
__device__ __forceinline__ uint8_t* slice_of(const QuantArgs& a, int pid, int kv, int h) {
  return a.pool + (size_t)pid * a.g.page + (size_t)a.layer * a.g.layer + (size_t)h * a.g.head + (size_t)kv * a.g.kv;
}
__device__ __forceinline__ float* scales_of(const QuantArgs& a, int pid, int kv, int h) {
  return a.scales + (size_t)pid * a.g.s_page + (size_t)a.layer * a.g.s_layer + (size_t)h * a.g.s_head +
         (size_t)kv * a.g.s_kv;
}

// Offset of (token t, dim d) inside a slice: K token-major, V tiled.
__device__ __forceinline__ int code_offset(int kv, int t, int d, int D) {
  return kv ? (((t >> 2) * 16 + (d & 15)) * (D >> 4) + (d >> 4)) * 4 + (t & 3) : t * D + d;
}

// int8, one wavefront per (token row, K/V, head).  src rows: [N][KH][D]
// (append) or [NP][KH][PS][D] (pages).  DMAX = 64, 128 or 256 >= D.
template <int SRC, int DMAX, bool PAGES>
__global__ void __launch_bounds__(64) quant_i8_kernel(QuantArgs a) {
  constexpr int PER = DMAX / 64;
  const int D = a.D, PS = a.PS;
  const int lane = threadIdx.x;
  const int kv = blockIdx.x / a.KH, h = blockIdx.x % a.KH;
  const int n = blockIdx.y;
  const int t = PAGES ? blockIdx.z : 0;
  const int pid = a.page_ids[n];
  const int slot = PAGES ? t : a.slots[n];
  if (pid < 0 || pid >= a.P || slot < 0 || slot >= PS) return;
  const bool valid = PAGES ? (t < a.slots[n]) : true;
  const void* src = kv ? a.value : a.key;
  const size_t row = PAGES ? (((size_t)n * a.KH + h) * PS + t) * D : ((size_t)n * a.KH + h) * D;
  float x[PER];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int d = i * 64 + lane;
    x[i] = (valid && d < D) ? load_src<SRC>(src, row + d) : 0.f;
    amax = fmaxf(amax, fabsf(x[i]));
  }
  amax = group_max<64>(amax);
  const float scale = __fdiv_rn(amax, 127.f);
  int8_t* dst = reinterpret_cast<int8_t*>(slice_of(a, pid, kv, h));
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int d = i * 64 + lane;
    if (d < D) dst[code_offset(kv, slot, d, D)] = int8_code(x[i], scale);
  }
  if (lane == 0) scales_of(a, pid, kv, h)[slot] = scale;
}

// ---------------------------------------------------------------------------
// Whole pages at D <= 128 from 16-byte aligned rows: one 256-thread workgroup
// per (page, K/V, head), a wavefront per group of four tokens in turn, lane
// (c, g) = lane % 16, lane / 16 with dims 8 c .. 8 c + 7 of token g of the
// group.  Sixteen lanes then cover a token's row in two (32-bit sources: four)
// 16-byte loads each, and the four tokens whose codes share a dword of the V
// tiling sit 16 lanes apart, where v_permlane swaps exchange them in
// registers.
// Bound: memory, once past the launch (about 5 us).  Against one row per
// wavefront with byte loads and stores: 512 pages of 8 heads x 16 x 128 from
// bf16 (51 MB) int8 40.9 -> 14.2 us, fp8 42.4 -> 13.4; 4096 pages int8 371 ->
// 87 us (4.6 TB/s), fp8 350 -> 82.
// ---------------------------------------------------------------------------

// x / s correctly rounded, from y = 1 / s correctly rounded: two residual
// corrections, the first of which brings the quotient within one ulp, where
// the second is exact (Markstein 1990).  Holds while the residuals stay
// normal: fast_scale below; for a smaller quotient (|x| < 2^-10 s at its
// smallest scale) both forms round to code 0 all the same.
__device__ __forceinline__ float div_by(float x, float s, float y) {
  float q = __fmul_rn(x, y);
  q = fmaf(fmaf(-q, s, x), y, q);
  return fmaf(fmaf(-q, s, x), y, q);
}
__device__ __forceinline__ bool fast_scale(float s) { return s > 0x1p-80f && s < 0x1p100f; }

// Four int8 codes, little end first: |q| <= 127 after the clamp, so adding
// 1.5 * 2^23 leaves the integer nearest to q (ties to even) in the low byte.
__device__ __forceinline__ uint32_t int8_codes4(const float* x, float s, float y) {
  uint32_t c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float q = fminf(fmaxf(div_by(x[i], s, y), -127.f), 127.f);
    c[i] = __float_as_uint(__fadd_rn(q, 12582912.f));
  }
  const uint32_t lo = __builtin_amdgcn_perm(c[1], c[0], 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm(c[3], c[2], 0x04000c0cu);
  return lo | hi;
}

__device__ __forceinline__ uint32_t pack4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return a | (b << 8) | (c << 16) | (d << 24);
}

// Codes of 8 elements, little end first.  v_cvt_pk_fp8_f32 gives
// vrm_e4m3::encode's code for every float up to 464 in magnitude (all of them
// compared) but not for NaN, whose codes are the only ones with seven low bits
// set: those lanes take the general path.
template <bool FP8>
__device__ __forceinline__ void codes8(const float (&x)[8], float scale, uint32_t& lo, uint32_t& hi) {
  bool slow = !fast_scale(scale);
  if (!slow) {
    const float y = __fdiv_rn(1.f, scale);
    if constexpr (FP8) {
      float q[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) q[i] = copysignf(div_by(x[i], scale, y), x[i]);  // -0 stays -0
      int a = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
      a = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], a, true);
      int b = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], 0, false);
      b = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], b, true);
      lo = (uint32_t)a;
      hi = (uint32_t)b;
      slow = ((((~lo & 0x7f7f7f7fu) - 0x01010101u) | ((~hi & 0x7f7f7f7fu) - 0x01010101u)) & 0x80808080u) != 0;
    } else {
      lo = int8_codes4(x, scale, y);
      hi = int8_codes4(x + 4, scale, y);
    }
  }
  if (slow) {
    uint32_t c[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) c[i] = FP8 ? fp8_code(x[i], scale) : (uint8_t)int8_code(x[i], scale);
    lo = pack4(c[0], c[1], c[2], c[3]);
    hi = pack4(c[4], c[5], c[6], c[7]);
  }
}

// First dims of a lane's two runs of four: 16-bit sources 8 c and 8 c + 4 (one
// 16-byte load), 32-bit ones 4 c and D / 2 + 4 c (two loads, each contiguous
// over the 16 lanes: 20 us against 33 us with adjacent ones at 512 pages).
template <int SRC>
__device__ __forceinline__ int run_dim(int c, int half, int D) {
  return SRC == VRM_SRC_F32 ? 4 * c + half * (D >> 1) : 8 * c + 4 * half;
}

template <int SRC>
__device__ __forceinline__ void load8(const void* p, size_t row, int c, int D, bool on, float (&x)[8]) {
  if constexpr (SRC == VRM_SRC_F32) {
    const float* q = static_cast<const float*>(p) + row;
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 a = on ? *reinterpret_cast<const float4*>(q + run_dim<SRC>(c, 0, D)) : z;
    const float4 b = on ? *reinterpret_cast<const float4*>(q + run_dim<SRC>(c, 1, D)) : z;
    x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w;
    x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
  } else {
    const uint4 z = make_uint4(0, 0, 0, 0);
    const uint4 d = on ? *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + row + 8 * c) : z;
    const uint32_t w[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t h = (w[k / 2] >> (16 * (k & 1))) & 0xffffu;
      x[k] = SRC == VRM_SRC_F16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
    }
  }
}

// Stores the codes (lo: the first run, hi: the second) of token 4 tg + g of a
// K slice, token-major.
template <int SRC>
__device__ __forceinline__ void store_k(uint8_t* dst, int tg, int c, int g, int D, bool on, uint32_t lo, uint32_t hi) {
  if (!on) return;
  uint8_t* row = dst + (size_t)(4 * tg + g) * D;
  if constexpr (SRC == VRM_SRC_F32) {
    *reinterpret_cast<uint32_t*>(row + run_dim<SRC>(c, 0, D)) = lo;
    *reinterpret_cast<uint32_t*>(row + run_dim<SRC>(c, 1, D)) = hi;
  } else {
    *reinterpret_cast<uint2*>(row + 8 * c) = make_uint2(lo, hi);
  }
}

// The same for a V slice, whose tiling puts four tokens of a dim in a dword:
// 4 x 4 byte transposes over the group's tokens.  After the first swap a lane
// holds one run of tokens 2 (g / 2) and 2 (g / 2) + 1, after the second two
// dims of all four.
template <int SRC>
__device__ __forceinline__ void store_v(uint32_t* tile, int tg, int c, int g, int D, bool on, uint32_t lo, uint32_t hi) {
  const auto s = __builtin_amdgcn_permlane16_swap(lo, hi, false, false);
  const uint32_t p = __builtin_amdgcn_perm(s[1], s[0], 0x05010400u);  // the run's dims 0, 1 of both tokens
  const uint32_t q = __builtin_amdgcn_perm(s[1], s[0], 0x07030602u);  // dims 2, 3
  const auto u = __builtin_amdgcn_permlane32_swap(p, q, false, false);
  if (on) {
    const int d = run_dim<SRC>(c, g & 1, D) + (g & 2);
    uint32_t* out = tile + (tg * 16 + (d & 15)) * (D >> 4) + (d >> 4);
    out[0] = __builtin_amdgcn_perm(u[1], u[0], 0x05040100u);
    out[D >> 4] = __builtin_amdgcn_perm(u[1], u[0], 0x07060302u);
  }
}

// Largest of the 16 lanes of a row (rotations within the row: every lane gets
// it).
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x122, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x121, 0xf, 0xf, false)));
  return v;
}

// A slice (page, K/V, head) goes to 4 / GROUPS wavefronts, GROUPS groups of
// four tokens in flight each.  With one wavefront per slice (GROUPS 4) V tiles
// leave through LDS in 1 KiB stores, and an fp8 page of up to 16 tokens needs
// no barrier for its maximum.
template <int SRC, int GROUPS, bool FP8>
__global__ void __launch_bounds__(256) quant_slices_kernel(QuantArgs a) {
  static_assert(!FP8 || GROUPS == 4, "an fp8 page's maximum is one wavefront's");
  constexpr int PER = 4 / GROUPS;  // wavefronts per slice
  __shared__ __align__(16) uint32_t v_lds[GROUPS > 1 ? 4 : 1][GROUPS > 1 ? GROUPS * 128 : 1];
  const int D = a.D, PS = a.PS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int s = blockIdx.x * GROUPS + wave / PER;
  if (s >= 2 * a.KH) return;
  const int kv = s / a.KH, h = s % a.KH;
  const int n = blockIdx.y;
  const int pid = a.page_ids[n];
  if (pid < 0 || pid >= a.P) return;
  const int n_valid = a.slots[n];
  const void* src = kv ? a.value : a.key;
  const size_t base = ((size_t)n * a.KH + h) * PS * D;
  uint8_t* dst = slice_of(a, pid, kv, h);
  float* sc = scales_of(a, pid, kv, h);
  const bool on = 8 * c < D;
  for (int tg0 = wave % PER * GROUPS; tg0 < PS / 4; tg0 += 4) {
    float x[GROUPS][8];
#pragma unroll
    for (int r = 0; r < GROUPS; ++r) {
      const int t = 4 * (tg0 + r) + g;
      load8<SRC>(src, base + (size_t)t * D, c, D, on && t < min(n_valid, PS), x[r]);
    }
    float page_scale = 0.f;
    if constexpr (FP8) {
      float amax = 0.f;
#pragma unroll
      for (int r = 0; r < GROUPS; ++r)
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[r][i]));
      page_scale = __fdiv_rn(group_max<64>(amax), 448.f);
      if (lane == 0) sc[0] = page_scale;
    }
#pragma unroll
    for (int r = 0; r < GROUPS; ++r) {
      if (GROUPS > 1 && tg0 + r >= PS / 4) break;
      float scale = page_scale;
      if constexpr (!FP8) {
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[r][i]));
        scale = __fdiv_rn(row16_max(amax), 127.f);
      }
      uint32_t lo = 0, hi = 0;
      if (scale > 0.f && (!FP8 || 4 * (tg0 + r) + g < n_valid)) codes8<FP8>(x[r], scale, lo, hi);
      if (kv == 0)
        store_k<SRC>(dst, tg0 + r, c, g, D, on, lo, hi);
      else if (GROUPS > 1)
        store_v<SRC>(v_lds[wave], r, c, g, D, on, lo, hi);
      else
        store_v<SRC>(reinterpret_cast<uint32_t*>(dst), tg0 + r, c, g, D, on, lo, hi);
      if (!FP8 && c == 0) sc[4 * (tg0 + r) + g] = scale;
    }
    if (GROUPS > 1 && kv == 1) {  // the groups' V tiles are one run of 4 D bytes each
      __syncwarp();
      uint4* out = reinterpret_cast<uint4*>(dst + (size_t)4 * tg0 * D);
      const int n16 = min(GROUPS, PS / 4 - tg0) * D / 4;
      for (int i = lane; i < n16; i += 64) out[i] = reinterpret_cast<const uint4*>(v_lds[wave])[i];
      __syncwarp();
    }
  }
}

// fp8: the page maximum first, its rows held in registers between (PS <= 16
// ROUNDS tokens).
template <int SRC, int ROUNDS>
__global__ void __launch_bounds__(256) quant_fp8_rows_kernel(QuantArgs a) {
  __shared__ float red[4];
  const int D = a.D, PS = a.PS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int kv = blockIdx.x / a.KH, h = blockIdx.x % a.KH;
  const int n = blockIdx.y;
  const int pid = a.page_ids[n];
  if (pid < 0 || pid >= a.P) return;
  const int n_valid = min(max(a.slots[n], 0), PS);
  const void* src = kv ? a.value : a.key;
  const size_t base = ((size_t)n * a.KH + h) * PS * D;
  const bool on = 8 * c < D;
  float x[ROUNDS][8];
  float amax = 0.f;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int t = 4 * (wave + 4 * r) + g;
    load8<SRC>(src, base + (size_t)t * D, c, D, on && t < n_valid, x[r]);
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[r][i]));
  }
  amax = group_max<64>(amax);
  if (lane == 0) red[wave] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float scale = __fdiv_rn(amax, 448.f);
  uint8_t* dst = slice_of(a, pid, kv, h);
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int tg = wave + 4 * r;
    if (tg < PS / 4) {
      uint32_t lo = 0, hi = 0;
      if (scale > 0.f && 4 * tg + g < n_valid) codes8<true>(x[r], scale, lo, hi);
      if (kv == 0)
        store_k<SRC>(dst, tg, c, g, D, on, lo, hi);
      else
        store_v<SRC>(reinterpret_cast<uint32_t*>(dst), tg, c, g, D, on, lo, hi);
    }
  }
  if (threadIdx.x == 0) *scales_of(a, pid, kv, h) = scale;
}

// fp8 whole pages, one 256-thread workgroup per (page, K/V, head): the page
// maximum over its valid tokens, then the codes (the source is read twice).
template <int SRC>
__global__ void __launch_bounds__(256) quant_fp8_pages_kernel(QuantArgs a) {
  const int D = a.D, PS = a.PS;
  const int N = PS * D;
  __shared__ float red[4];
  const int tid = threadIdx.x;
  const int kv = blockIdx.x / a.KH, h = blockIdx.x % a.KH;
  const int n = blockIdx.y;
  const int pid = a.page_ids[n];
  if (pid < 0 || pid >= a.P) return;
  const int n_valid = min(max(a.slots[n], 0), PS);
  const void* src = kv ? a.value : a.key;
  const size_t base = ((size_t)n * a.KH + h) * N;
  float amax = 0.f;
  for (int idx = tid; idx < n_valid * D; idx += 256) amax = fmaxf(amax, fabsf(load_src<SRC>(src, base + idx)));
  amax = group_max<64>(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float scale = __fdiv_rn(amax, 448.f);
  uint8_t* dst = slice_of(a, pid, kv, h);
  for (int idx = tid; idx < N; idx += 256) {
    const int t = idx / D, d = idx - t * D;
    dst[code_offset(kv, t, d, D)] = t < n_valid ? fp8_code(load_src<SRC>(src, base + idx), scale) : (uint8_t)0;
  }
  if (tid == 0) *scales_of(a, pid, kv, h) = scale;
}

// fp8 append, one 256-thread workgroup per (token, K/V, head).  The page
// scale only grows; when it does, the codes already in the page are
// re-encoded against the new scale.
template <int SRC>
__global__ void __launch_bounds__(256) quant_fp8_append_kernel(QuantArgs a) {
  const int D = a.D, PS = a.PS;  // D <= 256: one element per thread
  __shared__ float red[4];
  const int tid = threadIdx.x;
  const int kv = blockIdx.x / a.KH, h = blockIdx.x % a.KH;
  const int n = blockIdx.y;
  const int pid = a.page_ids[n];
  const int slot = a.slots[n];
  if (pid < 0 || pid >= a.P || slot < 0 || slot >= PS) return;
  const void* src = kv ? a.value : a.key;
  const size_t row = ((size_t)n * a.KH + h) * D;
  const float x = tid < D ? load_src<SRC>(src, row + tid) : 0.f;
  float amax = group_max<64>(fabsf(x));
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  float* const sp = scales_of(a, pid, kv, h);
  // Every thread reads the old scale before the barrier; thread 0 overwrites it after.
  const float old_scale = slot > 0 ? *sp : 0.f;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float want = __fdiv_rn(amax, 448.f);
  const float scale = fmaxf(old_scale, want);
  uint8_t* page = slice_of(a, pid, kv, h);
  if (slot > 0 && scale > old_scale) {
    for (int idx = tid; idx < slot * D; idx += 256) {
      const int off = code_offset(kv, idx / D, idx % D, D);
      const float y = e4m3fn_to_f32(page[off]) * old_scale;
      page[off] = fp8_code(y, scale);
    }
  }
  if (tid < D) page[code_offset(kv, slot, tid, D)] = fp8_code(x, scale);
  if (tid == 0) *sp = scale;
}

// Dequantize pages: out[n][2][KH][PS][D] float32.
template <bool FP8>
__global__ void __launch_bounds__(256) dequant_pages_kernel(QuantArgs a, float* out, int D) {
  const int kv = blockIdx.x / a.KH, h = blockIdx.x % a.KH;
  const int n = blockIdx.y;
  const int pid = a.page_ids[n];
  const size_t N = (size_t)a.PS * D;
  float* o = out + (((size_t)n * 2 + kv) * a.KH + h) * N;
  if (pid < 0 || pid >= a.P) {
    for (size_t i = threadIdx.x; i < N; i += 256) o[i] = 0.f;
    return;
  }
  const uint8_t* codes = slice_of(a, pid, kv, h);
  const float* sc = scales_of(a, pid, kv, h);
  for (size_t i = threadIdx.x; i < N; i += 256) {
    const int t = (int)(i / D), d = (int)(i % D);
    const uint8_t c = codes[code_offset(kv, t, d, D)];
    if (FP8) {
      o[i] = e4m3fn_to_f32(c) * sc[0];
    } else {
      o[i] = (float)(int8_t)c * sc[t];
    }
  }
}

int check_quant(const void* key, const void* value, int src_dtype, const int32_t* page_ids, const int32_t* slots,
                int n, void* pool, float* scales, int kv_dtype, int KH, int D, int PS, int L, int P, int layer,
                const char* who) {
  if (!key || !value || !page_ids || !slots || !pool || !scales) {
    set_error("%s: null pointer argument", who);
    return VRM_ERR_ARG;
  }
  if (n < 0 || KH <= 0 || D <= 0 || L <= 0 || P <= 0) {
    set_error("%s: bad sizes (N=%d KH=%d D=%d L=%d P=%d)", who, n, KH, D, L, P);
    return VRM_ERR_ARG;
  }
  if (layer < 0 || layer >= L) {
    set_error("%s: layer_idx %d outside [0, %d)", who, layer, L);
    return VRM_ERR_ARG;
  }
  if (src_dtype != VRM_SRC_F32 && src_dtype != VRM_SRC_F16 && src_dtype != VRM_SRC_BF16) {
    set_error("%s: unknown source dtype %d", who, src_dtype);
    return VRM_ERR_ARG;
  }
  if (!quant_pool(kv_dtype)) {
    set_error("%s: kv_dtype %d is not a quantized pool", who, kv_dtype);
    return VRM_ERR_ARG;
  }
  if (PS <= 0 || PS % 4 || PS > 65535) {
    set_error("%s: page_size %d unsupported (a positive multiple of 4)", who, PS);
    return VRM_ERR_UNSUPPORTED;
  }
  if (D % 16 || D > 256) {
    set_error("%s: head_dim %d unsupported (a multiple of 16 up to 256)", who, D);
    return VRM_ERR_UNSUPPORTED;
  }
  if (n > 65535 || 2 * KH > 65535) {
    set_error("%s: too many rows in one call (%d)", who, n);
    return VRM_ERR_UNSUPPORTED;
  }
  return check_pool_scales(kv_dtype, pool, scales, KH, PS, D, L, P, who);
}

// The row-group kernels: their lanes cover 128 dims, load 16 source bytes and
// store 8 code bytes at a time (every row and slice offset is a multiple of
// those; the buffers need to start on them), and the fp8 one holds at most 32
// tokens.
//
// From kManySlices (page, K/V, head) slices on, each has one wavefront (int8
// from bf16, four / one: 2048 slices 5.5 / 6.7 us, 4096 8.3 / 9.1, 8192 14.9 /
// 14.2, 16,384 26.0 / 22.7, 65,536 112 / 87; fp8 8192 15.7 / 13.4).
constexpr int kManySlices = 8192;
bool row_groups_ok(const QuantArgs& a, bool fp8) {
  const uintptr_t src = reinterpret_cast<uintptr_t>(a.key) | reinterpret_cast<uintptr_t>(a.value);
  return a.D <= 128 && (src & 15) == 0 && (reinterpret_cast<uintptr_t>(a.pool) & 15) == 0 && (!fp8 || a.PS <= 32);
}

template <int SRC, int DMAX>
void launch_quant(const QuantArgs& a, int n, int kv_dtype, bool pages, hipStream_t st) {
  if (pages && row_groups_ok(a, fp8_pool(kv_dtype))) {
    const dim3 grid(2 * a.KH, n), slices((2 * a.KH + 3) / 4, n);
    const bool many = (long long)n * 2 * a.KH >= kManySlices;
    if (!fp8_pool(kv_dtype)) {
      if (many)
        hipLaunchKernelGGL((quant_slices_kernel<SRC, 4, false>), slices, dim3(256), 0, st, a);
      else
        hipLaunchKernelGGL((quant_slices_kernel<SRC, 1, false>), grid, dim3(256), 0, st, a);
    } else if (a.PS <= 16) {
      if (many)
        hipLaunchKernelGGL((quant_slices_kernel<SRC, 4, true>), slices, dim3(256), 0, st, a);
      else
        hipLaunchKernelGGL((quant_fp8_rows_kernel<SRC, 1>), grid, dim3(256), 0, st, a);
    } else {
      hipLaunchKernelGGL((quant_fp8_rows_kernel<SRC, 2>), grid, dim3(256), 0, st, a);
    }
    return;
  }
  if (!fp8_pool(kv_dtype)) {
    if (pages)
      hipLaunchKernelGGL((quant_i8_kernel<SRC, DMAX, true>), dim3(2 * a.KH, n, a.PS), dim3(64), 0, st, a);
    else
      hipLaunchKernelGGL((quant_i8_kernel<SRC, DMAX, false>), dim3(2 * a.KH, n, 1), dim3(64), 0, st, a);
  } else {
    if (pages)
      hipLaunchKernelGGL((quant_fp8_pages_kernel<SRC>), dim3(2 * a.KH, n), dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((quant_fp8_append_kernel<SRC>), dim3(2 * a.KH, n), dim3(256), 0, st, a);
  }
}

template <int SRC>
void launch_quant_d(const QuantArgs& a, int n, int kv_dtype, bool pages, int D, hipStream_t st) {
  if (D <= 64)
    launch_quant<SRC, 64>(a, n, kv_dtype, pages, st);
  else if (D <= 128)
    launch_quant<SRC, 128>(a, n, kv_dtype, pages, st);
  else
    launch_quant<SRC, 256>(a, n, kv_dtype, pages, st);
}

int run_quant(const void* key, const void* value, int src_dtype, const int32_t* page_ids, const int32_t* slots,
              int n, void* pool, float* scales, int kv_dtype, int KH, int D, int PS, int L, int P, int layer,
              bool pages, vrm_stream_t stream, const char* who) {
  int rc = check_quant(key, value, src_dtype, page_ids, slots, n, pool, scales, kv_dtype, KH, D, PS, L, P, layer, who);
  if (rc) return rc;
  if (n == 0) {
    clear_error();
    return VRM_OK;
  }
  QuantArgs a{key, value, page_ids, slots, static_cast<uint8_t*>(pool), scales, KH, L, P, layer, D, PS,
              pool_geom(kv_dtype, KH, PS, D, D, P, L)};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  switch (src_dtype) {
    case VRM_SRC_F32: launch_quant_d<VRM_SRC_F32>(a, n, kv_dtype, pages, D, st); break;
    case VRM_SRC_F16: launch_quant_d<VRM_SRC_F16>(a, n, kv_dtype, pages, D, st); break;
    default: launch_quant_d<VRM_SRC_BF16>(a, n, kv_dtype, pages, D, st); break;
  }
  return launch_status(who);
}

}  // namespace
}  // namespace vrm

using namespace vrm;

extern "C" int vrm_kv_quant_append(const void* key, const void* value, int src_dtype, const int32_t* page_ids,
                                   const int32_t* slots, int N, void* kv_pool, float* kv_scales, int kv_dtype,
                                   int KH, int D, int PS, int L, int P, int layer_idx, vrm_stream_t stream) {
  return run_quant(key, value, src_dtype, page_ids, slots, N, kv_pool, kv_scales, kv_dtype, KH, D, PS, L, P,
                   layer_idx, false, stream, "vrm_kv_quant_append");
}

extern "C" int vrm_kv_quant_pages(const void* key, const void* value, int src_dtype, const int32_t* page_ids,
                                  const int32_t* n_valid, int NP, void* kv_pool, float* kv_scales, int kv_dtype,
                                  int KH, int D, int PS, int L, int P, int layer_idx, vrm_stream_t stream) {
  return run_quant(key, value, src_dtype, page_ids, n_valid, NP, kv_pool, kv_scales, kv_dtype, KH, D, PS, L, P,
                   layer_idx, true, stream, "vrm_kv_quant_pages");
}

extern "C" int vrm_kv_dequant_pages(const void* kv_pool, const float* kv_scales, int kv_dtype, const int32_t* page_ids,
                                    int NP, float* out, int KH, int D, int PS, int L, int P, int layer_idx,
                                    vrm_stream_t stream) {
  const char* who = "vrm_kv_dequant_pages";
  if (!kv_pool || !kv_scales || !page_ids || !out) {
    set_error("%s: null pointer argument", who);
    return VRM_ERR_ARG;
  }
  if (NP < 0 || NP > 65535 || KH <= 0 || 2 * KH > 65535 || D <= 0 || L <= 0 || P <= 0 || layer_idx < 0 ||
      layer_idx >= L) {
    set_error("%s: bad sizes", who);
    return VRM_ERR_ARG;
  }
  if (PS <= 0 || PS % 4 || D % 16 || D > 256) {
    set_error("%s: page_size %d / head_dim %d unsupported (multiples of 4 / 16)", who, PS, D);
    return VRM_ERR_UNSUPPORTED;
  }
  if (!quant_pool(kv_dtype)) {
    set_error("%s: kv_dtype %d is not a quantized pool", who, kv_dtype);
    return VRM_ERR_ARG;
  }
  const int rc = check_pool_scales(kv_dtype, kv_pool, kv_scales, KH, PS, D, L, P, who);
  if (rc) return rc;
  if (NP == 0) return VRM_OK;
  QuantArgs a{nullptr, nullptr, page_ids, nullptr, const_cast<uint8_t*>(static_cast<const uint8_t*>(kv_pool)),
              const_cast<float*>(kv_scales), KH, L, P, layer_idx, D, PS, pool_geom(kv_dtype, KH, PS, D, D, P, L)};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (fp8_pool(kv_dtype))
    hipLaunchKernelGGL(dequant_pages_kernel<true>, dim3(2 * KH, NP), dim3(256), 0, st, a, out, D);
  else
    hipLaunchKernelGGL(dequant_pages_kernel<false>, dim3(2 * KH, NP), dim3(256), 0, st, a, out, D);
  return launch_status(who);
}
