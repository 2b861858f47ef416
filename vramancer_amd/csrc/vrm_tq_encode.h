// Launchers of the TurboQuant kernels with 16 rows per wavefront: the encoder
// (vrm_tq_encode.hip) and decompression (vrm_tq_decompress.hip).
#pragma once
#include "vrm_common.h"

namespace vrm {

// Where the rows of a TurboQuant write come from and go to.  Pool writes
// (pool != nullptr) follow vrm_tq_layout.h's tuned layout; the others fill
// the codec's arrays, raw (angles [N][PD - 1], signs [N][PD / 2], one byte
// each) or packed (MSB first, angles [N][(PD - 1) bits / 8 rounded up], signs
// [N][PD / 16]).
struct TqEncodeArgs {
  const void* key;    // rows of head_dim elements (pool writes: the K side)
  const void* value;  // pool writes: the V side
  const int32_t* page_ids;
  const int32_t* slots;    // append: slot of each token; pages: nullptr
  const int32_t* n_valid;  // pages: valid tokens of each page; append: nullptr
  uint8_t* pool;
  int rows;  // rows of one side
  int KH, L, P, layer, bits, head_dim, padded_dim, src_dtype;
  int from_pool;  // pages: key/value are a float pool [P][L][2][KH][16][head_dim] read at (page_ids[n], layer)
  int packed;     // codec arrays: packed bytes
  const float* signs;
  const float* jl;
  const float* lut;
  uint16_t* radius;
  uint8_t* angles;
  uint8_t* qjl_signs;
  uint16_t* qjl_norms;
};

// Rows to decompress: angles [N][PD - 1] bytes, or packed (MSB first, 4-byte
// aligned); out [N][head_dim], or the rotated rows [N][PD].
struct TqDecompressArgs {
  const uint16_t* radius;
  const uint8_t* angles;
  int N, head_dim, padded_dim, bits;
  int packed, rotated;
  const float* signs;
  const float* lut;
  float* out;
};

// True for the settings these kernels serve: padded dim 64 or 128, 2 to 4
// bits per angle; the encoder also wants padded_dim / 2 QJL rows.
inline bool tq_rows_ok(int padded_dim, int bits) {
  return (padded_dim == 64 || padded_dim == 128) && bits >= 2 && bits <= 4;
}
inline bool tq_tile_ok(int padded_dim, int bits, int qjl_dim) {
  return tq_rows_ok(padded_dim, bits) && qjl_dim == padded_dim / 2;
}

// The caller checks launch_status.
void launch_tq_encode(const TqEncodeArgs& a, hipStream_t stream);
void launch_tq_decompress(const TqDecompressArgs& a, hipStream_t stream);

}  // namespace vrm
