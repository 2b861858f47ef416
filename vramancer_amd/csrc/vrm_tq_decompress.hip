// TurboQuant decompression, 16 rows per wavefront (padded dim 64 or 128, 2 to
// 4 bits per angle), from raw or packed angles.
//
// A lane rebuilds its quarter of a row from the radius down: the product chain
// of the two top levels, then a tree of 2 x 2, 4, ... multiplications by the
// {cos, sin} of each angle, the reference's products in its order, then the
// inverse rotation in registers.  One launch reads the packed bits; unpacking
// them to bytes first moved 127 bytes a row through memory three times.
// Bound: a mix of vector issue, LDS reads (angle table, bins) and the output's
// stores.  65,536 rows of 128 at 3 bits, packed: unpacking (angles 22 us, signs
// 9 us) and one row per wavefront (24 us) -> 10.7 us (37 MB at 3.4 TB/s); raw
// angles 23.4 -> 16.4 us, their bytes read one by one from LDS.
#include "vrm_tq_bin.h"
#include "vrm_tq_encode.h"
#include "vrm_tq_row.h"
#include "vrm_tq_tile.h"

namespace vrm {
namespace {

#pragma clang fp contract(off)

constexpr int kWavesPerWg = 4;

template <int BITS, int PD, bool PACKED>
__global__ void __launch_bounds__(64 * kWavesPerWg) tq_decompress_tile_kernel(TqDecompressArgs a) {
  constexpr int NQ = PD / 4, LQ = PD == 128 ? 4 : 3, NB = 1 << BITS;
  constexpr int RW = ((PD - 1) * BITS + 31) / 32;              // dwords of a packed row
  constexpr int ROWB = PACKED ? RW * 4 : PD - 1;               // bytes of a row
  constexpr int STAGE = (kTile * ROWB + 8 + 15) / 16 * 16;     // reads run up to two dwords past a run
  __shared__ __align__(16) uint8_t stage_lds[kWavesPerWg][STAGE];
  constexpr int OUTW = PD + 4;  // row stride of the output tile: 16 rows on distinct banks
  __shared__ __align__(16) float out_lds[kWavesPerWg][kTile * OUTW];
  __shared__ float2 cs[2 * NB];  // {level 0, levels >= 1} x bins: {cos, sin}
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  if (threadIdx.x < 2 * NB) {
    const int half = threadIdx.x / NB, i = threadIdx.x % NB;
    cs[threadIdx.x] = make_float2(a.lut[half * 2 * NB + i], a.lut[half * 2 * NB + NB + i]);
  }
  __syncthreads();  // the workgroup's only barrier, before any wavefront leaves
  const long long n0 = ((long long)blockIdx.x * kWavesPerWg + wave) * kTile;
  if (n0 >= a.N) return;
  const int nrows = (int)min((long long)kTile, a.N - n0);
  uint8_t* stage = stage_lds[wave];
  const uint8_t* src = a.angles + (size_t)n0 * ROWB;
  const int total = nrows * ROWB;
  if (PACKED || (reinterpret_cast<uintptr_t>(src) & 3) == 0) {
    for (int i = lane; i < total / 4; i += 64) {
      const uint32_t x = reinterpret_cast<const uint32_t*>(src)[i];
      reinterpret_cast<uint32_t*>(stage)[i] = PACKED ? __builtin_bswap32(x) : x;
    }
    if (lane < (total & 3)) stage[(total & ~3) + lane] = src[(total & ~3) + lane];
  } else {
    for (int i = lane; i < total; i += 64) stage[i] = src[i];
  }
  const int row = min(r, nrows - 1);  // lanes past the last row repeat it and store nothing
  const float radius = f16_bits_to_f32(a.radius[n0 + row]);
  row_sync();

  const uint8_t* bytes = stage + row * ROWB;
  const uint32_t* words = reinterpret_cast<const uint32_t*>(stage) + row * RW;
  // level-major bins first .. first + 63 / BITS, left-aligned (packed)
  auto run_at = [&](int first) {
    const int pos = first * BITS, sh = pos & 31;
    const uint32_t* p = words + (pos >> 5);
    const uint64_t x = ((uint64_t)p[0] << 32) | p[1];
    return sh ? (x << sh) | (p[2] >> (32 - sh)) : x;
  };
  auto bin_at = [&](int b) -> uint32_t {
    if constexpr (PACKED) return (uint32_t)(run_at(b) >> (64 - BITS));
    return min((uint32_t)bytes[b], (uint32_t)(NB - 1));  // caller-supplied bins stay in the table
  };
  float v[NQ];
  {
    const float2 f1 = cs[NB + bin_at(PD - 2)], f0 = cs[NB + bin_at(tq::level_offset(PD, LQ + 1) + (g >> 1))];
    v[0] = __fmul_rn(__fmul_rn(radius, g & 2 ? f1.y : f1.x), g & 1 ? f0.y : f0.x);
  }
#pragma unroll
  for (int l = LQ; l >= 0; --l) {
    const int first = tq::level_offset(PD, l) + (NQ >> (l + 1)) * g;
    uint64_t run = 0;
    if constexpr (PACKED) run = run_at(first);
#pragma unroll
    for (int i = (NQ >> (l + 1)) - 1; i >= 0; --i) {  // downwards: v[i] is read before v[2 i], v[2 i + 1] are written
      const uint32_t b = PACKED ? (uint32_t)(run >> (64 - BITS * (i + 1))) & (NB - 1) : bin_at(first + i);
      const float2 f = cs[(l == 0 ? 0 : NB) + b];
      const float x = v[i];
      v[2 * i] = __fmul_rn(x, f.x);
      v[2 * i + 1] = __fmul_rn(x, f.y);
    }
  }
  const int e0 = NQ * g;
  const int width = a.rotated ? PD : a.head_dim;
  if (!a.rotated) {
    tile_fwht<PD>(v);
    // the fast division wants finite, ordinary values: radii that are (codes
    // shrink a row by at most 10^7, sums of it cancel to a 2^-24th of that)
    if (PD == 64) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) v[i] = __fmul_rn(v[i], 0.125f);
    } else if (__ballot(!(radius > 0.f && radius < 65536.f)) == 0) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) v[i] = vrm_tq_bin::div_sqrt128(v[i]);
    } else {
      const float root = (float)sqrt((double)PD);
#pragma unroll
      for (int i = 0; i < NQ; ++i) v[i] = __fdiv_rn(v[i], root);
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i) v[i] = __fmul_rn(v[i], a.signs[e0 + i]);
  }
  if (width == PD && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0) {
    // whole rows: through LDS, so that a store instruction writes 1 KiB in one
    // piece (a lane's own 16 bytes lie PD floats from its neighbour's: 16.0
    // against 10.7 us at 65,536 rows)
    float* t = out_lds[wave];
#pragma unroll
    for (int c = 0; c < NQ / 4; ++c)
      *reinterpret_cast<float4*>(t + r * OUTW + e0 + 4 * c) =
          make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
    row_sync();
    float4* dst = reinterpret_cast<float4*>(a.out + (size_t)n0 * PD);
#pragma unroll
    for (int k = 0; k < kTile * PD / 256; ++k) {
      const int i = k * 64 + lane, row_i = i / (PD / 4);
      if (row_i < nrows) dst[i] = *reinterpret_cast<const float4*>(t + row_i * OUTW + i % (PD / 4) * 4);
    }
    return;
  }
  if (r >= nrows) return;
  float* out = a.out + (size_t)(n0 + r) * width + e0;
  if (((reinterpret_cast<uintptr_t>(a.out) | (uintptr_t)(width * 4)) & 15) == 0) {
#pragma unroll
    for (int c = 0; c < NQ / 4; ++c)
      if (e0 + 4 * c < width)
        reinterpret_cast<float4*>(out)[c] = make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
  } else {
#pragma unroll
    for (int i = 0; i < NQ; ++i)
      if (e0 + i < width) out[i] = v[i];
  }
}

template <int BITS, int PD>
void launch_rows(const TqDecompressArgs& a, hipStream_t st) {
  const long long tiles = ((long long)a.N + kTile - 1) / kTile;
  const dim3 grid((unsigned)((tiles + kWavesPerWg - 1) / kWavesPerWg));
  if (a.packed)
    hipLaunchKernelGGL((tq_decompress_tile_kernel<BITS, PD, true>), grid, dim3(64 * kWavesPerWg), 0, st, a);
  else
    hipLaunchKernelGGL((tq_decompress_tile_kernel<BITS, PD, false>), grid, dim3(64 * kWavesPerWg), 0, st, a);
}

}  // namespace

void launch_tq_decompress(const TqDecompressArgs& a, hipStream_t st) {
#define VRM_TQ_ROWS(B)                 \
  if (a.padded_dim == 64)              \
    launch_rows<B, 64>(a, st);         \
  else                                 \
    launch_rows<B, 128>(a, st)
  switch (a.bits) {
    case 2: VRM_TQ_ROWS(2); break;
    case 3: VRM_TQ_ROWS(3); break;
    default: VRM_TQ_ROWS(4); break;
  }
#undef VRM_TQ_ROWS
}

}  // namespace vrm
