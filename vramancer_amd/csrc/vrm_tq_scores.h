// Launchers shared by the TurboQuant score and sparse-attention entries
// (vrm_tq_sparse.hip, vrm_sparse_attend.hip).
#pragma once
#include "vrm_common.h"

namespace vrm {

// Compressed rows in the codec's raw format.
struct TqCodes {
  const uint16_t* radius;
  const uint8_t* angles;     // [N][padded_dim - 1]
  const uint8_t* qjl_signs;  // keys: [N][qjl_dim]
  const uint16_t* qjl_norms; // keys: [N]
};

// What the selection leaves of a row of scores for the weighted sum: token n
// is kept when its key is above t_key, or equals it and n <= last_tie.
struct TopkRow {
  uint32_t t_key;
  int last_tie;
  float max;
  int pad;
};

// Longest row the one-pass selection holds in registers.
constexpr int kMaxSelectRow = 32768;

// Ascending float order <-> ascending unsigned order.
__device__ __forceinline__ uint32_t order_key(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Selects the k largest scores of each row of N <= kMaxSelectRow, one workgroup
// per row.
void launch_topk_select(const float* scores, int M, int N, long long ld, int k, TopkRow* rows, hipStream_t st);

// Query features ws [M][padded_dim + qjl_dim]: the rotated query, then its JL
// projection.
void launch_tq_query(const float* q, int M, int head_dim, int padded_dim, const float* signs, const float* jl,
                     int qjl_dim, float* ws, hipStream_t st);

// scores[m][n] = out_scale (q_rot[m] . k_polar[n] + QJL correction) on the
// matrix cores, from query features ws [M][padded_dim + qjl_dim]; padded_dim
// 64 or 128, qjl_dim half of it, bits <= 4, code arrays aligned to 4 (angles)
// and 16 bytes (signs), ws to 16.
bool tq_score_tiles_ok(const TqCodes& k, int padded_dim, int qjl_dim, int bits, const float* ws);
void launch_tq_score_tiles(const float* ws, int M, const TqCodes& k, int N, int padded_dim, const float* lut, int bits,
                           float coef, float out_scale, float* scores, hipStream_t st);

}  // namespace vrm
