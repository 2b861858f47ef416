// TurboQuant scores and sparse-V attention on compressed rows (padded dim 64
// or 128, qjl_dim half of it, up to 4 bits per angle).
//
// Scores (tq_score_tile_kernel): [keys x F] x [F x queries] on
// v_mfma_f32_16x16x4_f32, F = padded_dim + qjl_dim features (the polar
// reconstruction, then coef norm (2 sign - 1)).  Lane (r, g) = lane % 16,
// lane / 16 rebuilds quarter g of key r, so its 32 (16) values are features of
// k index g and need no exchange; the query features are staged in LDS once
// per 128 keys.
//
// Sparse V (tq_sparse_pv_kernel): the reference keeps each row's k largest
// weights; across a group of query rows nearly every token is kept by some, so
// the weighted sum runs over all tokens on the matrix cores, with weight 0
// where a row dropped the token.  The values are rebuilt in registers from
// their codes, in the rotated space: the rotation is linear and is undone once
// per output row (tq_sparse_out_kernel).  Lane (c, t) of a wavefront rebuilds
// dims PD / 16 c .. of tokens 4 t .. 4 t + 3, which is the operand layout of
// the product: no value row goes through memory.
//
// 40 query rows, 32,768 keys at 3 bits, top 10 %: scores 20.4 -> 14.7 us;
// decompression (11), compaction (25) and gathered sum (26 + 4) -> 18.1 + 5.7 us;
// the whole call 173 -> 63 us.  None is near a unit's peak: each is a chain of
// staging, table look-ups and products over one or two wavefronts per SIMD.
#include "vrm_tq_row.h"
#include "vrm_tq_scores.h"
#include "vrm_tq_tile.h"

#include <algorithm>

namespace vrm {
namespace {

#pragma clang fp contract(off)

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRowBlock = 48;     // query rows whose features are staged together
constexpr int kScoreWaves = 8;    // 16 keys each
constexpr int kPvWaves = 4;

// {cos, sin} of every bin, level 0 then levels >= 1: [2][nb] at 2 nb <= 32.
__device__ __forceinline__ void stage_table(float2* cs, const float* lut, int nb, int tid) {
  if (tid < 2 * nb) {
    const int half = tid / nb, i = tid % nb;
    cs[tid] = make_float2(lut[half * 2 * nb + i], lut[half * 2 * nb + nb + i]);
  }
}

// Copies this wavefront's rows (n0 a multiple of 16, so their bytes start on
// the array's 4-byte alignment) into LDS.
__device__ __forceinline__ void stage_rows(uint8_t* stage, const uint8_t* src, int total, int lane) {
  for (int i = lane; i < total / 4; i += 64)
    reinterpret_cast<uint32_t*>(stage)[i] = reinterpret_cast<const uint32_t*>(src)[i];
  if (lane < (total & 3)) stage[(total & ~3) + lane] = src[(total & ~3) + lane];
}

template <int PD>
__global__ void __launch_bounds__(64 * kScoreWaves) tq_score_tile_kernel(const float* ws, int M, TqCodes k, int N,
                                                                       const float* lut, int bits, float coef,
                                                                       float out_scale, float* scores) {
  constexpr int QJ = PD / 2, F = PD + QJ, NQ = PD / 4, LQ = PD == 128 ? 4 : 3;
  constexpr int J = F / 4;             // features of a lane: NQ polar, QJ / 4 signs
  constexpr int QW = F + 4;            // LDS stride of a query row: 16 rows on distinct banks
  constexpr int ROWB = PD - 1;
  __shared__ __align__(16) float q_lds[kRowBlock * QW];
  __shared__ __align__(16) uint8_t bins_lds[kScoreWaves][kTile * ROWB + 16];
  __shared__ float2 cs[32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int nb = 1 << bits;
  stage_table(cs, lut, nb, threadIdx.x);
  const int n0 = (blockIdx.x * kScoreWaves + wave) * kTile;
  const int nk = max(0, min(kTile, N - n0));  // 0: the wavefront only joins the barriers
  uint8_t* bins = bins_lds[wave];
  auto stage_queries = [&](int m0, int rows) {
    for (int i = threadIdx.x; i < rows * (F / 4); i += 64 * kScoreWaves) {
      const int m = i / (F / 4), f = i - m * (F / 4);
      *reinterpret_cast<float4*>(q_lds + m * QW + 4 * f) = reinterpret_cast<const float4*>(ws + (size_t)(m0 + m) * F)[f];
    }
  };
  if (nk) stage_rows(bins, k.angles + (size_t)n0 * ROWB, nk * ROWB, lane);
  stage_queries(0, min(kRowBlock, M));
  __syncthreads();
  const int key = min(n0 + r, N - 1);
  float A[J];
  if (nk) {
    const uint8_t* kb = bins + min(r, nk - 1) * ROWB;
    auto factor = [&](int level, int angle) {
      return cs[(level == 0 ? 0 : nb) + min((int)kb[tq::level_offset(PD, level) + angle], nb - 1)];
    };
    const float2 f1 = factor(LQ + 2, 0), f0 = factor(LQ + 1, g >> 1);
    A[0] = __fmul_rn(__fmul_rn(f16_bits_to_f32(k.radius[key]), g & 2 ? f1.y : f1.x), g & 1 ? f0.y : f0.x);
#pragma unroll
    for (int l = LQ; l >= 0; --l) {
#pragma unroll
      for (int i = (NQ >> (l + 1)) - 1; i >= 0; --i) {  // downwards: A[i] is read before A[2 i], A[2 i + 1] are written
        const float2 f = factor(l, (NQ >> (l + 1)) * g + i);
        const float x = A[i];
        A[2 * i] = __fmul_rn(x, f.x);
        A[2 * i + 1] = __fmul_rn(x, f.y);
      }
    }
    const float cn = __fmul_rn(coef, f16_bits_to_f32(k.qjl_norms[key]));
    const uint32_t* sg = reinterpret_cast<const uint32_t*>(k.qjl_signs + (size_t)key * QJ + QJ / 4 * g);
#pragma unroll
    for (int t = 0; t < QJ / 16; ++t) {
      const uint32_t w = sg[t];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float s = (float)((w >> (8 * u)) & 0xffu);
        A[NQ + 4 * t + u] = __fmul_rn(__fsub_rn(__fmul_rn(s, 2.f), 1.f), cn);
      }
    }
  }
  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(scores) & 15) == 0;
  for (int m0 = 0; m0 < M; m0 += kRowBlock) {
    const int rows = min(kRowBlock, M - m0);
    if (m0) {
      __syncthreads();
      stage_queries(m0, rows);
      __syncthreads();
    }
    if (!nk) continue;
    for (int mt = 0; mt < rows; mt += 16) {
      const float* qb = q_lds + min(mt + r, rows - 1) * QW;
      v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < J / 4; ++t) {
        const int f = 4 * t < NQ ? NQ * g + 4 * t : PD + QJ / 4 * g + 4 * t - NQ;
        const float4 b = *reinterpret_cast<const float4*>(qb + f);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[4 * t], b.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[4 * t + 1], b.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[4 * t + 2], b.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[4 * t + 3], b.w, acc, 0, 0, 0);
      }
      // C[key 4 g + i][query row]
      if (mt + r < rows) {
        float* out = scores + (size_t)(m0 + mt + r) * N + n0 + 4 * g;
        if (vec && 4 * g + 4 <= nk) {
          *reinterpret_cast<float4*>(out) = make_float4(__fmul_rn(acc[0], out_scale), __fmul_rn(acc[1], out_scale),
                                                        __fmul_rn(acc[2], out_scale), __fmul_rn(acc[3], out_scale));
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (4 * g + i < nk) out[i] = __fmul_rn(acc[i], out_scale);
        }
      }
    }
  }
}

// Partial sums part[blockIdx.x][m][PD] and weight sums part_sum[blockIdx.x][m],
// m over the rows of blockIdx.y's block of 16 MT, of the workgroup's 64 tokens.
template <int PD, int MT>
__global__ void __launch_bounds__(64 * kPvWaves) tq_sparse_pv_kernel(const float* scores, int M, int N,
                                                                   const TopkRow* rows, TqCodes v, const float* lut,
                                                                   int bits, float* part, float* part_sum) {
  constexpr int DPL = PD / 16;                 // dims of a lane
  constexpr int LL = PD == 128 ? 3 : 2;        // levels below its node
  constexpr int NL = PD == 128 ? 7 : 6;
  constexpr int ROWB = PD - 1;
  __shared__ __align__(16) uint8_t bins_lds[kPvWaves][kTile * ROWB + 16];
  __shared__ float2 cs[32];
  __shared__ __align__(16) float fold[2][MT * 16 * PD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, t = lane >> 4;
  const int nb = 1 << bits;
  stage_table(cs, lut, nb, threadIdx.x);
  __syncthreads();
  const int m0 = blockIdx.y * 16 * MT;
  TopkRow row[MT];
  const float* srow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = min(m0 + 16 * i + c, M - 1);
    row[i] = rows[m];
    srow[i] = scores + (size_t)m * N;
  }
  v4f acc[MT][DPL];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int d = 0; d < DPL; ++d) acc[i][d] = v4f{0.f, 0.f, 0.f, 0.f};
  __shared__ float sum_lds[kPvWaves][MT * 16];
  float wsum[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) wsum[i] = 0.f;
  uint8_t* bins = bins_lds[wave];
  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(scores) & 15) == 0;
  const int n0 = (blockIdx.x * kPvWaves + wave) * kTile;
  if (n0 < N) {
    const int nk = min(kTile, N - n0);
    stage_rows(bins, v.angles + (size_t)n0 * ROWB, nk * ROWB, lane);
    float s4[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (vec && 4 * t + 4 <= nk) {
        const float4 x = *reinterpret_cast<const float4*>(srow[i] + n0 + 4 * t);
        s4[i][0] = x.x, s4[i][1] = x.y, s4[i][2] = x.z, s4[i][3] = x.w;
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) s4[i][s] = 4 * t + s < nk ? srow[i][n0 + 4 * t + s] : 0.f;
      }
    }
    row_sync();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int tok = 4 * t + s, tk = min(tok, nk - 1), n = n0 + tok;
      const uint8_t* kb = bins + tk * ROWB;
      auto factor = [&](int level, int angle) {
        return cs[(level == 0 ? 0 : nb) + min((int)kb[tq::level_offset(PD, level) + angle], nb - 1)];
      };
      float x[DPL];
      // a value row without finite numbers reaches the rows that keep it and
      // no others (0 times it would be NaN): weight NaN over zeros
      const float radius = f16_bits_to_f32(v.radius[n0 + tk]);
      const bool finite = fabsf(radius) < INFINITY;
      x[0] = finite ? radius : 0.f;
#pragma unroll
      for (int l = NL - 1; l >= LL; --l) {
        const float2 f = factor(l, c >> (l + 1 - LL));
        x[0] = __fmul_rn(x[0], (c >> (l - LL)) & 1 ? f.y : f.x);
      }
#pragma unroll
      for (int l = LL - 1; l >= 0; --l) {
#pragma unroll
        for (int i = (DPL >> (l + 1)) - 1; i >= 0; --i) {
          const float2 f = factor(l, (DPL >> (l + 1)) * c + i);
          const float y = x[i];
          x[2 * i] = __fmul_rn(y, f.x);
          x[2 * i + 1] = __fmul_rn(y, f.y);
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const uint32_t key = order_key(s4[i][s]);
        const bool keep = tok < nk && (key > row[i].t_key || (key == row[i].t_key && n <= row[i].last_tie));
        const float w = keep ? (finite ? expf(s4[i][s] - row[i].max) : NAN) : 0.f;
        wsum[i] += w;
#pragma unroll
        for (int d = 0; d < DPL; ++d) acc[i][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, x[d], acc[i][d], 0, 0, 0);
      }
    }
  }
  // the four wavefronts' sums, two by two; lane (c, t) holds rows 4 t + j of
  // each tile at dims DPL c + d
  auto put = [&](float* f) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int d = 0; d < DPL; d += 4)
          *reinterpret_cast<float4*>(f + (16 * i + 4 * t + j) * PD + DPL * c + d) =
              make_float4(acc[i][d][j], acc[i][d + 1][j], acc[i][d + 2][j], acc[i][d + 3][j]);
  };
  auto add = [&](const float* f) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int d = 0; d < DPL; ++d) acc[i][d][j] += f[(16 * i + 4 * t + j) * PD + DPL * c + d];
  };
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const float w = strided_sum<16>(wsum[i]);
    if (t == 0) sum_lds[wave][16 * i + c] = w;
  }
  if (wave >= 2) put(fold[wave - 2]);
  __syncthreads();
  if (wave < 2) add(fold[wave]);
  if (wave == 1) put(fold[1]);
  __syncthreads();
  if (wave == 0) {
    if (lane < 16 * MT && m0 + lane < M) {
      float w = 0.f;
#pragma unroll
      for (int i = 0; i < kPvWaves; ++i) w += sum_lds[i][lane];
      part_sum[(size_t)blockIdx.x * M + m0 + lane] = w;
    }
    add(fold[1]);
    float* dst = part + ((size_t)blockIdx.x * M + m0) * PD;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (m0 + 16 * i + 4 * t + j < M)
#pragma unroll
          for (int d = 0; d < DPL; d += 4)
            *reinterpret_cast<float4*>(dst + (16 * i + 4 * t + j) * PD + DPL * c + d) =
                make_float4(acc[i][d][j], acc[i][d + 1][j], acc[i][d + 2][j], acc[i][d + 3][j]);
  }
}

// out[m][head_dim] = unrotate(sum of the partials / weight sum): one
// 1024-thread workgroup per row.
template <int PD>
__global__ void __launch_bounds__(1024) tq_sparse_out_kernel(const float* part, const float* part_sum, int blocks,
                                                           int M, int head_dim, const float* signs, float* out) {
  constexpr int C = PD / 4, G = 1024 / C, PER = tq_per_lane(PD);
  __shared__ __align__(16) float sum_lds[G][PD];
  __shared__ float l_lds[16];
  const int m = blockIdx.x, d = threadIdx.x % C, s = threadIdx.x / C;
  const float4* src = reinterpret_cast<const float4*>(part + (size_t)m * PD) + d;
  const size_t stride = (size_t)M * C;
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int b = s; b < blocks; b += G) {
    const float4 x = src[b * stride];
    sum = make_float4(sum.x + x.x, sum.y + x.y, sum.z + x.z, sum.w + x.w);
  }
  *reinterpret_cast<float4*>(&sum_lds[s][4 * d]) = sum;
  float l = 0.f;
  for (int b = threadIdx.x; b < blocks; b += 1024) l += part_sum[(size_t)b * M + m];
  l = group_sum<64>(l);
  if ((threadIdx.x & 63) == 0) l_lds[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  const float root = (float)sqrt((double)PD);
  l = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) l += l_lds[i];
  float v[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < G; ++i) x += sum_lds[i][k * 64 + lane];
    v[k] = x / l;
  }
  fwht<PD>(v, lane);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = k * 64 + lane;
    if (e < head_dim) out[(size_t)m * head_dim + e] = v[k] / root * signs[e];
  }
}

}  // namespace

bool tq_score_tiles_ok(const TqCodes& k, int padded_dim, int qjl_dim, int bits, const float* ws) {
  return (padded_dim == 64 || padded_dim == 128) && qjl_dim == padded_dim / 2 && bits <= 4 &&
         ((reinterpret_cast<uintptr_t>(k.angles) & 3) | (reinterpret_cast<uintptr_t>(k.qjl_signs) & 15) |
          (reinterpret_cast<uintptr_t>(ws) & 15)) == 0;
}

void launch_tq_score_tiles(const float* ws, int M, const TqCodes& k, int N, int padded_dim, const float* lut, int bits,
                           float coef, float out_scale, float* scores, hipStream_t st) {
  const dim3 grid((unsigned)((N + (long long)kScoreWaves * kTile - 1) / (kScoreWaves * kTile)));
  if (padded_dim == 64)
    hipLaunchKernelGGL(tq_score_tile_kernel<64>, grid, dim3(64 * kScoreWaves), 0, st, ws, M, k, N, lut, bits, coef,
                       out_scale, scores);
  else
    hipLaunchKernelGGL(tq_score_tile_kernel<128>, grid, dim3(64 * kScoreWaves), 0, st, ws, M, k, N, lut, bits, coef,
                       out_scale, scores);
}

}  // namespace vrm

using namespace vrm;

namespace {

// Workgroups of the weighted sum: 16 tokens per wavefront (32: fewer partials,
// but 19.2 us against 18.1 at 32,768 tokens).
int pv_blocks(int N) { return (N + kPvWaves * kTile - 1) / (kPvWaves * kTile); }

struct SparseWs {
  int rows;                              // query rows of one pass
  size_t scores, sel, sum, part, total;  // byte offsets; the query features come first
};
// Query rows are taken in passes whose scores and partial sums (padded_dim / 64
// times the scores) stay within kPassBytes, so that the workspace does not grow
// with M: 4096 rows over 32,768 keys took 1.6 GB, 65,535 rows 26.  Smaller
// passes leave compute units without a row to select (1024 rows over 32,768
// keys in one pass 545 us, in passes of 672 rows 560, of 144 740).  A pass is a
// multiple of the 48 rows that the sum takes at once.
constexpr size_t kPassBytes = (size_t)256 << 20;
SparseWs sparse_ws(int M, int N, int padded_dim, int qjl_dim) {
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  const size_t row = ((size_t)N + padded_dim + qjl_dim + (size_t)pv_blocks(N) * (padded_dim + 1)) * sizeof(float);
  SparseWs w{};
  w.rows = (int)std::min<size_t>((size_t)M, std::max<size_t>(kPassBytes / row / 48, 1) * 48);
  w.scores = up((size_t)w.rows * (padded_dim + qjl_dim) * sizeof(float));
  w.sel = w.scores + up((size_t)w.rows * N * sizeof(float));
  w.sum = w.sel + up((size_t)w.rows * sizeof(TopkRow));
  w.part = w.sum + up((size_t)pv_blocks(N) * w.rows * sizeof(float));
  w.total = w.part + (size_t)pv_blocks(N) * w.rows * padded_dim * sizeof(float);
  return w;
}

template <int PD>
void launch_pv(const float* scores, int M, int N, const TopkRow* rows, const TqCodes& v, const float* lut, int bits,
               int head_dim, const float* signs, float* part, float* part_sum, float* out, hipStream_t st) {
  const int blocks = pv_blocks(N);
  const dim3 wg(64 * kPvWaves);
  if (M <= 16)
    hipLaunchKernelGGL((tq_sparse_pv_kernel<PD, 1>), dim3(blocks, 1), wg, 0, st, scores, M, N, rows, v, lut, bits,
                       part, part_sum);
  else if (M <= 32)
    hipLaunchKernelGGL((tq_sparse_pv_kernel<PD, 2>), dim3(blocks, 1), wg, 0, st, scores, M, N, rows, v, lut, bits,
                       part, part_sum);
  else
    hipLaunchKernelGGL((tq_sparse_pv_kernel<PD, 3>), dim3(blocks, (M + 47) / 48), wg, 0, st, scores, M, N, rows, v,
                       lut, bits, part, part_sum);
  hipLaunchKernelGGL(tq_sparse_out_kernel<PD>, dim3(M), dim3(1024), 0, st, part, part_sum, blocks, M,
                     head_dim, signs, out);
}

}  // namespace

extern "C" size_t vrm_turboquant_sparse_attend_workspace_bytes(int M, int N, int padded_dim, int qjl_dim) {
  if (M < 0 || N <= 0 || padded_dim <= 0 || qjl_dim <= 0) return 0;
  return sparse_ws(M, N, padded_dim, qjl_dim).total;
}

extern "C" int vrm_turboquant_sparse_attend(const float* q, int M, const uint16_t* k_radius, const uint8_t* k_angles,
                                            const uint8_t* k_signs, const uint16_t* k_norms,
                                            const uint16_t* v_radius, const uint8_t* v_angles, int N, int k,
                                            int head_dim, int padded_dim, int n_levels, int bits, int qjl_dim,
                                            const float* signs, const float* jl, const float* angle_lut, float scale,
                                            void* workspace, size_t workspace_bytes, float* out,
                                            vrm_stream_t stream) {
  const char* who = "vrm_turboquant_sparse_attend";
  if (M < 0 || M > 65535 || N <= 0 || k < 1 || k > N || head_dim <= 0 || head_dim > padded_dim) {
    set_error("%s: bad sizes (M=%d N=%d k=%d head_dim=%d padded_dim=%d)", who, M, N, k, head_dim, padded_dim);
    return VRM_ERR_ARG;
  }
  if ((padded_dim != 64 && padded_dim != 128) || (1 << n_levels) != padded_dim || qjl_dim != padded_dim / 2 ||
      bits < 1 || bits > 4 || N > kMaxSelectRow) {
    set_error("%s: serves padded_dim 64 or 128, qjl_dim half of it, 1 to 4 bits and up to %d rows (got %d, %d, %d, %d)",
              who, kMaxSelectRow, padded_dim, qjl_dim, bits, N);
    return VRM_ERR_UNSUPPORTED;
  }
  if (M == 0) {
    clear_error();
    return VRM_OK;
  }
  if (!q || !k_radius || !k_angles || !k_signs || !k_norms || !v_radius || !v_angles || !signs || !jl || !angle_lut ||
      !workspace || !out) {
    set_error("%s: null pointer argument", who);
    return VRM_ERR_ARG;
  }
  const SparseWs w = sparse_ws(M, N, padded_dim, qjl_dim);
  if (workspace_bytes < w.total) {
    set_error("%s: workspace of %zu bytes, need %zu", who, workspace_bytes, w.total);
    return VRM_ERR_WORKSPACE;
  }
  uint8_t* base = static_cast<uint8_t*>(workspace);
  float* feat = static_cast<float*>(workspace);
  const TqCodes keys{k_radius, k_angles, k_signs, k_norms};
  if (!tq_score_tiles_ok(keys, padded_dim, qjl_dim, bits, feat) || (reinterpret_cast<uintptr_t>(v_angles) & 3)) {
    set_error("%s: angles must be aligned to 4 bytes, signs and workspace to 16", who);
    return VRM_ERR_ARG;
  }
  float* scores = reinterpret_cast<float*>(base + w.scores);
  TopkRow* rows = reinterpret_cast<TopkRow*>(base + w.sel);
  float* part = reinterpret_cast<float*>(base + w.part);
  float* part_sum = reinterpret_cast<float*>(base + w.sum);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const TqCodes vals{v_radius, v_angles, nullptr, nullptr};
  for (int m0 = 0; m0 < M; m0 += w.rows) {
    const int m = std::min(w.rows, M - m0);
    launch_tq_query(q + (size_t)m0 * head_dim, m, head_dim, padded_dim, signs, jl, qjl_dim, feat, st);
    launch_tq_score_tiles(feat, m, keys, N, padded_dim, angle_lut, bits, (float)(sqrt(M_PI / 2.0) / qjl_dim), scale,
                          scores, st);
    launch_topk_select(scores, m, N, N, k, rows, st);
    float* o = out + (size_t)m0 * head_dim;
    if (padded_dim == 64)
      launch_pv<64>(scores, m, N, rows, vals, angle_lut, bits, head_dim, signs, part, part_sum, o, st);
    else
      launch_pv<128>(scores, m, N, rows, vals, angle_lut, bits, head_dim, signs, part, part_sum, o, st);
  }
  return launch_status(who);
}
