// TurboQuant encoder, 16 rows per wavefront (padded dim 64 or 128, 2 to 4
// bits per angle, padded_dim / 2 QJL rows): the pool's page writes and the
// codec's compress.
//
// Lane (r, g) = lane % 16, lane / 16 holds the quarter of row r over dims
// PD / 4 * g ...: the subtree whose angles the page layout keeps together, and
// the k-slice a lane feeds to v_mfma_f32_16x16x32_bf16.  So the butterflies
// below h = PD / 4, the radii and angles of the lower levels, the polar decode
// and the record of a quarter are register work of one lane with 16 or 32
// independent chains, and only the two top levels cross lanes (v_permlane
// swaps).
//
// What bounds it: vector issue (memory traffic takes a fifth of its time).
// Measured at padded dim 128, 3 bits, bf16, against one row per wavefront with
// the IEEE, fdlibm and float64 sequences: 65,536 K and 65,536 V rows into pages
// 409 -> 38 us, 65,536 rows through the codec 236 -> 28 us.  The work per value
// is kept down by
//   * angle bins by polynomial, with the defining path only for rows that
//     have an angle at a sector edge (vrm_tq_bin.h; 0.2 % of rows at 3 bits);
//   * the rotation's division as multiply and two fused corrections, and the
//     square root as v_rsq_f32 with one fused correction (equal to sqrtf for
//     every float from 1e-12 up);
//   * QJL products on the matrix cores: residual and JL matrix as bf16 hi + lo
//     pairs, three products.  Only the sign of a dot product is kept, and it
//     is taken from there when the value exceeds the bound of the products'
//     error; otherwise (about 3e-4 of the signs) the dot product is taken in
//     float64, and if that is within its own rounding of zero, by the
//     defining chain.
// Codes are those of vrm_tq_row.h bit for bit.
#include "vrm_tq_encode.h"

#include "vrm_tq_bin.h"
#include "vrm_tq_row.h"
#include "vrm_tq_tile.h"

namespace vrm {
namespace {

#pragma clang fp contract(off)

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// Correctly rounded square root of x >= 1e-12: the radii carry that floor.
__device__ __forceinline__ float sqrt_radius(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const float g = __fmul_rn(x, y);
  return fmaf(fmaf(-g, g, x), __fmul_rn(0.5f, y), g);
}

__device__ __forceinline__ float radius_of(float x0, float x1) {
  return sqrt_radius(__fadd_rn(__fadd_rn(__fmul_rn(x0, x0), __fmul_rn(x1, x1)), 1e-12f));
}

__device__ __forceinline__ float load_any(int src, const void* p, size_t i) {
  return src == VRM_SRC_F32 ? load_row<VRM_SRC_F32>(p, i)
                            : src == VRM_SRC_F16 ? load_row<VRM_SRC_F16>(p, i) : load_row<VRM_SRC_BF16>(p, i);
}

// LDS of a workgroup: the JL matrix as bf16 hi and lo fragments, its longest
// row's 2-norm, the angle table, and a scratch row per wavefront.
template <int PD>
struct TileLds {
  static constexpr int QJL = PD / 2;
  static constexpr int CT = QJL / 16;      // 16-row tiles of the JL matrix
  static constexpr int KS = PD / 32;       // k-steps
  static constexpr int FRAGS = CT * KS * 2 * 64;  // 16-byte fragments: (tile, k-step, hi / lo, lane)
  static constexpr size_t frag_bytes = (size_t)FRAGS * 16;
  static constexpr size_t fixed_bytes = frag_bytes + QJL * 4 + 64 * 8;
  // a RowLds, or the 16 rows' codec output
  static constexpr size_t wave_bytes = (sizeof(RowLds<PD>) > 16 * PD ? sizeof(RowLds<PD>) : 16 * PD) + 64;
};

// Splits 8 floats into bf16 hi (nearest) and the bf16 of the remainder.
__device__ __forceinline__ void split8(const float (&x)[8], v8bf& hi, v8bf& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const __bf16 h = (__bf16)x[i];
    hi[i] = h;
    lo[i] = (__bf16)__fsub_rn(x[i], (float)h);
  }
}

// Bound of |mfma dot - exact dot| over ||residual|| ||jl row||: the operands'
// representation 2^-18 each and the dropped lo * lo 2^-18, together below
// 2^-16.4, and 128 additions of hi * hi terms, each rounded (or cut) at
// 2^-23 of at most sum |r| |j|: 2^-16; the cross terms' sums are 2^-8 of
// those.  Together below 2^-15.1.
constexpr float kSignBound = 3.2e-5f;  // 2^-14.93

template <int BITS, int PD>
__global__ void __launch_bounds__(512) tq_encode_tile_kernel(TqEncodeArgs a, int tiles_per_wg) {
  using Q = Quarter<PD, BITS>;
  using S = TileLds<PD>;
  constexpr int NQ = Q::NQ, LQ = Q::LQ, QJL = S::QJL, NB = 1 << BITS;
  extern __shared__ __align__(16) uint8_t lds[];
  v8bf* frags = reinterpret_cast<v8bf*>(lds);
  float* jl_norm2 = reinterpret_cast<float*>(lds + S::frag_bytes);
  float2* cs = reinterpret_cast<float2*>(lds + S::frag_bytes + QJL * 4);  // [2][NB] {cos, sin}
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  uint8_t* scratch = lds + S::fixed_bytes + (size_t)wave * S::wave_bytes;
  RowLds<PD>& w = *reinterpret_cast<RowLds<PD>*>(scratch);
  const bool to_pool = a.pool != nullptr;
  const int kv = blockIdx.y;  // codec: 0

  if (kv == 0) {  // values carry no QJL fields
    if (threadIdx.x < QJL) jl_norm2[threadIdx.x] = 0.f;
    if (threadIdx.x < 2 * NB) {
      const int half = threadIdx.x / NB, i = threadIdx.x % NB;
      cs[threadIdx.x] = make_float2(a.lut[half * 2 * NB + i], a.lut[half * 2 * NB + NB + i]);
    }
    __syncthreads();
    const bool jl_vec = (reinterpret_cast<uintptr_t>(a.jl) & 15) == 0;
#pragma unroll 4
    for (int i = threadIdx.x; i < S::CT * S::KS * 64; i += blockDim.x) {
      const int l = i & 63, ks = (i >> 6) % S::KS, ct = (i >> 6) / S::KS;
      const int j = 16 * ct + (l & 15);
      const float* src = a.jl + (size_t)j * PD + NQ * (l >> 4) + 8 * ks;
      float x[8];
      float n2 = 0.f;
      if (jl_vec) {
        const float4 u = reinterpret_cast<const float4*>(src)[0], v = reinterpret_cast<const float4*>(src)[1];
        x[0] = u.x, x[1] = u.y, x[2] = u.z, x[3] = u.w;
        x[4] = v.x, x[5] = v.y, x[6] = v.z, x[7] = v.w;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = src[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) n2 = fmaf(x[e], x[e], n2);
      v8bf hi, lo;
      split8(x, hi, lo);
      frags[((ct * S::KS + ks) * 2 + 0) * 64 + l] = hi;
      frags[((ct * S::KS + ks) * 2 + 1) * 64 + l] = lo;
      atomicAdd(&jl_norm2[j], n2);
    }
    __syncthreads();  // the last barrier: wavefronts leave independently below
  }

  const int tile = blockIdx.x * tiles_per_wg + wave;
  if (wave >= tiles_per_wg || tile >= (a.rows + kTile - 1) / kTile) return;
  const int x_row = tile * kTile + r;
  const int x = min(x_row, a.rows - 1);  // rows past the end repeat the last one and store nothing

  // where the row comes from and goes to
  bool store = x_row < a.rows, live = true;
  size_t src_first = (size_t)x * a.head_dim;
  uint8_t* slice = nullptr;
  int t = 0;
  if (to_pool) {
    int n, h;
    if (a.slots) {
      n = x / a.KH;
      h = x - n * a.KH;
      t = a.slots[n];
    } else {
      t = x % tq::kTokens;
      const int nh = x / tq::kTokens;
      n = nh / a.KH;
      h = nh - n * a.KH;
      live = t < a.n_valid[n];
    }
    const int pid = a.page_ids[n];
    const bool inside = pid >= 0 && pid < a.P && t >= 0 && t < tq::kTokens;
    store = store && inside;  // rows aimed outside the pool are dropped
    live = live && inside;
    const size_t at = (((size_t)(inside ? pid : 0) * a.L + a.layer) * 2 + kv) * a.KH + h;
    if (a.from_pool) src_first = (at * tq::kTokens + t) * a.head_dim;
    slice = a.pool + at * tq::slice_bytes(PD, BITS);
  }
  if (__ballot(store) == 0) return;
  const void* src = kv ? a.value : a.key;

  Q q;
#pragma unroll
  for (int i = 0; i < Q::WORDS; ++i) q.w[i] = 0;
  float radius = 0.f, norm = 0.f;
  uint32_t sign_word = 0;  // lanes g < QJL / 32: QJL signs 32 g .. 32 g + 31 of row r

  const bool work = store && live;
  if (__ballot(work) != 0) {
    float v[NQ];
    // ---- load and rotate ----
    {
      const int esize = a.src_dtype == VRM_SRC_F32 ? 4 : 2;
      const bool vec = ((reinterpret_cast<uintptr_t>(src) | (uintptr_t)(a.head_dim * esize)) & 15) == 0;
      const int e0 = NQ * g;
      if (!vec) {
#pragma unroll
        for (int i = 0; i < NQ; ++i)
          v[i] = work && e0 + i < a.head_dim ? load_any(a.src_dtype, src, src_first + e0 + i) : 0.f;
      } else if (a.src_dtype == VRM_SRC_F32) {
        const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(src) + src_first + e0);
#pragma unroll
        for (int c = 0; c < NQ / 4; ++c) {
          const float4 f = work && e0 + 4 * c < a.head_dim ? p[c] : make_float4(0.f, 0.f, 0.f, 0.f);
          v[4 * c] = f.x;
          v[4 * c + 1] = f.y;
          v[4 * c + 2] = f.z;
          v[4 * c + 3] = f.w;
        }
      } else {
        const v4u* p = reinterpret_cast<const v4u*>(static_cast<const uint16_t*>(src) + src_first + e0);
        v4u d[NQ / 8];
#pragma unroll
        for (int c = 0; c < NQ / 8; ++c) d[c] = work && e0 + 8 * c < a.head_dim ? p[c] : v4u{0, 0, 0, 0};
        if (a.src_dtype == VRM_SRC_F16) {
#pragma unroll
          for (int i = 0; i < NQ; ++i) v[i] = f16_bits_to_f32((d[i / 8][i % 8 / 2] >> (16 * (i & 1))) & 0xffffu);
        } else {
#pragma unroll
          for (int i = 0; i < NQ; ++i)
            v[i] = __uint_as_float(i & 1 ? d[i / 8][i % 8 / 2] & 0xffff0000u : d[i / 8][i % 8 / 2] << 16);
        }
      }
      const float4* sg = reinterpret_cast<const float4*>(a.signs + e0);
      if ((reinterpret_cast<uintptr_t>(a.signs) & 15) == 0) {
#pragma unroll
        for (int c = 0; c < NQ / 4; ++c) {
          const float4 f = sg[c];
          v[4 * c] = __fmul_rn(v[4 * c], f.x);
          v[4 * c + 1] = __fmul_rn(v[4 * c + 1], f.y);
          v[4 * c + 2] = __fmul_rn(v[4 * c + 2], f.z);
          v[4 * c + 3] = __fmul_rn(v[4 * c + 3], f.w);
        }
      } else {
#pragma unroll
        for (int i = 0; i < NQ; ++i) v[i] = __fmul_rn(v[i], a.signs[e0 + i]);
      }
    }
    tile_fwht<PD>(v);
#pragma unroll
    for (int i = 0; i < NQ; ++i) v[i] = PD == 64 ? __fmul_rn(v[i], 0.125f) : vrm_tq_bin::div_sqrt128(v[i]);

    // ---- radii and angles ----
    bool edge = false;
    uint32_t bin_a, bin_b;  // level LQ + 1 of this half, the root
    {
      float child[NQ];
#pragma unroll
      for (int i = 0; i < NQ; ++i) child[i] = v[i];
#pragma unroll
      for (int l = 0; l <= LQ; ++l) {
#pragma unroll
        for (int i = 0; i < (NQ >> (l + 1)); ++i) {
          const float x0 = child[2 * i], x1 = child[2 * i + 1];
          const float rcp = __builtin_amdgcn_rcpf(fmaxf(fabsf(x0), fabsf(x1)));
          bool e;
          const int b = l == 0 ? vrm_tq_bin::fast_bin<BITS, true>(x0, x1, rcp, e)
                               : vrm_tq_bin::fast_bin<BITS, false>(x0, x1, rcp, e);
          edge = edge || e;
          q.put(slot_in_quarter<PD, BITS>(l, i), (uint32_t)b);
          child[i] = radius_of(x0, x1);
        }
      }
      bool e;
      float o = xor_shfl<16>(child[0]);
      float x0 = g & 1 ? o : child[0], x1 = g & 1 ? child[0] : o;
      bin_a = (uint32_t)vrm_tq_bin::fast_bin<BITS, false>(x0, x1, __builtin_amdgcn_rcpf(fmaxf(x0, x1)), e);
      edge = edge || e;
      const float half = radius_of(x0, x1);
      o = xor_shfl<32>(half);
      x0 = g & 2 ? o : half;
      x1 = g & 2 ? half : o;
      bin_b = (uint32_t)vrm_tq_bin::fast_bin<BITS, false>(x0, x1, __builtin_amdgcn_rcpf(fmaxf(x0, x1)), e);
      edge = edge || e;
      radius = radius_of(x0, x1);
    }
    edge = edge || !(radius < 0x1p60f);  // NaN, infinite or huge rows
    // rows with an angle at a sector edge: the defining path
    uint64_t redo = __ballot(edge && work);
    redo = (redo | (redo >> 16) | (redo >> 32) | (redo >> 48)) & 0xffffu;
    while (redo) {
      const int row = __builtin_ctzll(redo);
      redo &= redo - 1;
      const uint64_t first = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(src_first >> 32), row) << 32) |
                             (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)src_first, row);
      float vr[tq_per_lane(PD)];
      const float rad = encode_row<PD>([&](int e) { return load_any(a.src_dtype, src, first + e); }, a.head_dim, a.signs,
                                       BITS, vr, w, lane);
      if (r == row) {
#pragma unroll
        for (int i = 0; i < Q::WORDS; ++i) q.w[i] = 0;
#pragma unroll
        for (int l = 0; l <= LQ; ++l)
#pragma unroll
          for (int i = 0; i < (NQ >> (l + 1)); ++i)
            q.put(slot_in_quarter<PD, BITS>(l, i), w.bins[tq::level_offset(PD, l) + (NQ >> (l + 1)) * g + i]);
        bin_a = w.bins[tq::level_offset(PD, LQ + 1) + (g >> 1)];
        bin_b = w.bins[PD - 2];
        radius = rad;
#pragma unroll
        for (int i = 0; i < NQ; ++i) v[i] = w.rot[NQ * g + i];
      }
      row_sync();  // the next row reuses the scratch
    }
    q.put(NQ - 1, g == 0 ? bin_b : g == 3 ? 0u : bin_a);

    // ---- QJL residual, signs and norm ----
    if (kv == 0) {
      float* dump = reinterpret_cast<float*>(scratch);
      {
        float rec[NQ];
        const float2 f6 = cs[NB + bin_b], f5 = cs[NB + bin_a];
        rec[0] = __fmul_rn(__fmul_rn(radius, g & 2 ? f6.y : f6.x), g & 1 ? f5.y : f5.x);
#pragma unroll
        for (int l = LQ; l >= 0; --l) {
#pragma unroll
          for (int i = (NQ >> (l + 1)) - 1; i >= 0; --i) {  // downwards: rec[i] is read before rec[2 i], rec[2 i + 1]
            const float2 f = cs[(l == 0 ? 0 : NB) + q.get(slot_in_quarter<PD, BITS>(l, i))];
            const float x0 = rec[i];
            rec[2 * i] = __fmul_rn(x0, f.x);
            rec[2 * i + 1] = __fmul_rn(x0, f.y);
          }
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i) v[i] = __fsub_rn(v[i], rec[i]);
      }
      // norm: eight fused accumulators over e % 8, in element order, so they
      // pass from quarter to quarter
      {
        float acc[8];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            float c = s == 0 ? 0.f
                             : __int_as_float(__builtin_amdgcn_ds_bpermute((lane - 16) << 2, __float_as_int(acc[k])));
#pragma unroll
            for (int m = 0; m < NQ / 8; ++m) c = fmaf(v[8 * m + k], v[8 * m + k], c);
            acc[k] = c;
          }
        }
        float s = acc[0];
#pragma unroll
        for (int k = 1; k < 8; ++k) s = __fadd_rn(s, acc[k]);
        s = __int_as_float(__builtin_amdgcn_ds_bpermute((48 + r) << 2, __float_as_int(s)));
        norm = sqrt_rn(s);
      }
      v8bf rh[S::KS], rl[S::KS];
#pragma unroll
      for (int ks = 0; ks < S::KS; ++ks) {
        float x8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x8[e] = v[8 * ks + e];
        split8(x8, rh[ks], rl[ks]);
      }
      float jmax2 = 0.f;
#pragma unroll
      for (int j = 0; j < QJL / 16; ++j) jmax2 = fmaxf(jmax2, jl_norm2[16 * j + r]);
      jmax2 = group_max<16>(jmax2);
      const float jmax = sqrt_rn(jmax2);
      // below 2^-90 the operands' bf16 parts could leave the normal range
      const float bound = norm > 0x1p-90f && jmax > 0x1p-90f ? kSignBound * norm * jmax : INFINITY;
      uint32_t pos = 0, near = 0;  // bit 4 ct + i: sign j = 16 ct + 4 g + i of row r
#pragma unroll
      for (int ct = 0; ct < S::CT; ++ct) {
        v4f hh = {0.f, 0.f, 0.f, 0.f}, cross = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < S::KS; ++ks) {
          const v8bf jh = frags[((ct * S::KS + ks) * 2 + 0) * 64 + lane];
          const v8bf jlo = frags[((ct * S::KS + ks) * 2 + 1) * 64 + lane];
          hh = __builtin_amdgcn_mfma_f32_16x16x32_bf16(jh, rh[ks], hh, 0, 0, 0);
          cross = __builtin_amdgcn_mfma_f32_16x16x32_bf16(jh, rl[ks], cross, 0, 0, 0);
          cross = __builtin_amdgcn_mfma_f32_16x16x32_bf16(jlo, rh[ks], cross, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float d = hh[i] + cross[i];
          pos |= d > 0.f ? 1u << (4 * ct + i) : 0u;
          near |= !(fabsf(d) > bound) ? 1u << (4 * ct + i) : 0u;
        }
      }
      near = work ? near : 0u;
      uint64_t todo = __ballot(near != 0);
      while (todo) {
        const int l0 = __builtin_ctzll(todo);
        todo &= todo - 1;
        uint32_t bits = (uint32_t)__builtin_amdgcn_readlane((int)near, l0);
        row_sync();
        if (r == (l0 & 15)) {
#pragma unroll
          for (int i = 0; i < NQ; ++i) dump[NQ * g + i] = v[i];
        }
        row_sync();
        const float n_row = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(norm), l0));
        while (bits) {
          const int b = __builtin_ctz(bits);
          bits &= bits - 1;
          const float* jr = a.jl + (size_t)(16 * (b >> 2) + 4 * (l0 >> 4) + (b & 3)) * PD;
          double s = 0.0;
#pragma unroll
          for (int k = 0; k < PD / 64; ++k) s = fma((double)dump[64 * k + lane], (double)jr[64 * k + lane], s);
#pragma unroll
          for (int m = 1; m < 64; m <<= 1) {
            const int lo = __builtin_amdgcn_ds_bpermute((lane ^ m) << 2, __double2loint(s));
            const int hi = __builtin_amdgcn_ds_bpermute((lane ^ m) << 2, __double2hiint(s));
            s += __hiloint2double(hi, lo);
          }
          // both this sum and the defining chain are within 2^-45 of the
          // norms' product of the exact dot product
          if (!(fabs(s) > 0x1p-43 * (double)n_row * (double)jmax)) {
            s = 0.0;
            for (int e = 0; e < PD; ++e) s = fma((double)dump[e], (double)jr[e], s);
          }
          if (lane == l0) pos = s > 0.0 ? pos | (1u << b) : pos & ~(1u << b);
        }
        row_sync();
      }
      // lane g's nibbles of each word, gathered over the row's four lanes
      uint32_t words[QJL / 32];
#pragma unroll
      for (int k = 0; k < QJL / 32; ++k) {
        uint32_t x32 = (((pos >> (8 * k)) & 15u) << (4 * g)) | (((pos >> (8 * k + 4)) & 15u) << (16 + 4 * g));
        x32 |= __float_as_uint(xor_shfl<16>(__uint_as_float(x32)));
        x32 |= __float_as_uint(xor_shfl<32>(__uint_as_float(x32)));
        words[k] = x32;
      }
      sign_word = QJL == 32 || g == 0 ? words[0] : words[QJL / 32 - 1];
    }
    if (to_pool && !live) {  // zero records below
#pragma unroll
      for (int i = 0; i < Q::WORDS; ++i) q.w[i] = 0;
      radius = 0.f;
      norm = 0.f;
      sign_word = 0;
    }
  }

  if (to_pool) {
    if (!store) return;
    uint8_t* rec = slice + (size_t)t * tq::angle_bytes(PD, BITS);
    if constexpr (PD == 128) {
      uint32_t* dst = reinterpret_cast<uint32_t*>(rec) + g * BITS;
#pragma unroll
      for (int i = 0; i < BITS; ++i) dst[i] = q.w[i];
    } else {  // 16 slots: BITS half-words per quarter
      uint16_t* dst = reinterpret_cast<uint16_t*>(rec) + g * BITS;
#pragma unroll
      for (int i = 0; i < BITS; ++i) dst[i] = (uint16_t)(q.w[i / 2] >> (16 * (i & 1)));
    }
    if (g == 0) reinterpret_cast<uint16_t*>(slice + tq::radius_offset(PD, BITS))[t] = f32_to_f16_bits(radius);
    if (kv == 0) {
      if (g < QJL / 32)
        reinterpret_cast<uint32_t*>(slice + tq::signs_offset(PD, BITS) + t * tq::sign_bytes(PD))[g] = sign_word;
      if (g == 3) reinterpret_cast<uint16_t*>(slice + tq::norms_offset(PD, BITS))[t] = f32_to_f16_bits(norm);
    }
    return;
  }

  // ---- codec arrays ----
  const int n0 = tile * kTile, nrows = min(kTile, a.rows - n0);
  const uint32_t spare = q.get(NQ - 1);
  const int la = tq::level_offset(PD, LQ + 1);
  row_sync();
  if (a.packed) {
    // level-major bit stream, most significant bit first: each lane ORs its
    // runs (contiguous within a level) into the row's big-endian dwords
    constexpr int RW = ((PD - 1) * BITS + 31) / 32;
    uint32_t* st = reinterpret_cast<uint32_t*>(scratch);
    for (int i = lane; i < kTile * RW; i += 64) st[i] = 0;
    row_sync();
    uint32_t* row = st + r * RW;
    auto put_run = [&](uint64_t run, int bitpos, int len) {  // run: len bits, left-aligned in 64
      const int sh = bitpos & 31, wd = bitpos >> 5;
      const uint64_t x64 = run >> sh;
      atomicOr(&row[wd], (uint32_t)(x64 >> 32));
      if (sh + len > 32) atomicOr(&row[wd + 1], (uint32_t)x64);
      if (sh + len > 64) atomicOr(&row[wd + 2], (uint32_t)((run << (64 - sh)) >> 32));
    };
#pragma unroll
    for (int l = 0; l <= LQ; ++l) {
      uint64_t run = 0;
#pragma unroll
      for (int i = 0; i < (NQ >> (l + 1)); ++i)
        run |= (uint64_t)q.get(slot_in_quarter<PD, BITS>(l, i)) << (64 - BITS * (i + 1));
      put_run(run, (tq::level_offset(PD, l) + (NQ >> (l + 1)) * g) * BITS, (NQ >> (l + 1)) * BITS);
    }
    // spares: lane 0 the root, lanes 1 and 2 the two angles below it
    if (g < 3) put_run((uint64_t)spare << (64 - BITS), (g == 0 ? PD - 2 : la + g - 1) * BITS, BITS);
    row_sync();
    uint32_t* dst = reinterpret_cast<uint32_t*>(a.angles) + (size_t)n0 * RW;
    for (int i = lane; i < nrows * RW; i += 64) dst[i] = __builtin_bswap32(st[i]);
    if (store && g < QJL / 32)
      reinterpret_cast<uint32_t*>(a.qjl_signs)[(size_t)x * (QJL / 32) + g] = __builtin_bswap32(__brev(sign_word));
  } else {
    uint8_t* row = scratch + r * (PD - 1);
#pragma unroll
    for (int l = 0; l <= LQ; ++l)
#pragma unroll
      for (int i = 0; i < (NQ >> (l + 1)); ++i)
        row[tq::level_offset(PD, l) + (NQ >> (l + 1)) * g + i] = (uint8_t)q.get(slot_in_quarter<PD, BITS>(l, i));
    if (g < 3) row[g == 0 ? PD - 2 : la + g - 1] = (uint8_t)spare;
    row_sync();
    const int total = nrows * (PD - 1);
    uint8_t* dst = a.angles + (size_t)n0 * (PD - 1);
    if ((reinterpret_cast<uintptr_t>(dst) & 3) == 0) {
      for (int i = lane; i < total / 4; i += 64)
        reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(scratch)[i];
      if (lane < (total & 3)) dst[(total & ~3) + lane] = scratch[(total & ~3) + lane];
    } else {
      for (int i = lane; i < total; i += 64) dst[i] = scratch[i];
    }
    // sign bytes: this lane's QJL / 4 of the row, from the word that holds them
    if (store) {
      constexpr int PER = QJL / 4;
      const uint32_t wd = (uint32_t)__builtin_amdgcn_ds_bpermute((((PER * g) >> 5) * 16 + r) << 2, (int)sign_word);
      uint8_t* sd = a.qjl_signs + (size_t)x * QJL + PER * g;
      const uint32_t bits = wd >> ((PER * g) & 31);
      if ((reinterpret_cast<uintptr_t>(a.qjl_signs) & 3) == 0) {
#pragma unroll
        for (int i = 0; i < PER / 4; ++i) {
          const uint32_t nib = (bits >> (4 * i)) & 15u;
          reinterpret_cast<uint32_t*>(sd)[i] =
              (nib & 1u) | ((nib & 2u) << 7) | ((nib & 4u) << 14) | ((nib & 8u) << 21);
        }
      } else {
#pragma unroll
        for (int i = 0; i < PER; ++i) sd[i] = (uint8_t)((bits >> i) & 1u);
      }
    }
  }
  if (store && g == 0) a.radius[x] = f32_to_f16_bits(radius);
  if (store && g == 3) a.qjl_norms[x] = f32_to_f16_bits(norm);
}

template <int BITS, int PD>
void launch_tile(const TqEncodeArgs& a, hipStream_t st) {
  using S = TileLds<PD>;
  const int tiles = (a.rows + kTile - 1) / kTile;
  // Many rows: 8 tiles share a workgroup's staged JL matrix.  Few: they spread
  // over the compute units first, and the wavefronts without a tile only help
  // with the staging.
  const int per_wg = tiles >= 2048 ? 8 : tiles >= 512 ? 4 : tiles >= 256 ? 2 : 1;
  const int waves = per_wg > 4 ? per_wg : 4;
  const size_t lds = S::fixed_bytes + (size_t)per_wg * S::wave_bytes;
  hipLaunchKernelGGL((tq_encode_tile_kernel<BITS, PD>), dim3((tiles + per_wg - 1) / per_wg, a.pool ? 2 : 1),
                     dim3(64 * waves), lds, st, a, per_wg);
}

}  // namespace

void launch_tq_encode(const TqEncodeArgs& a, hipStream_t st) {
#define VRM_TQ_TILE(B)                 \
  if (a.padded_dim == 64)              \
    launch_tile<B, 64>(a, st);         \
  else                                 \
    launch_tile<B, 128>(a, st)
  switch (a.bits) {
    case 2: VRM_TQ_TILE(2); break;
    case 3: VRM_TQ_TILE(3); break;
    default: VRM_TQ_TILE(4); break;
  }
#undef VRM_TQ_TILE
}

}  // namespace vrm
