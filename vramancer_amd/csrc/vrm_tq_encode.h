// Launchers of the TurboQuant tile encoder (vrm_tq_encode.hip).
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

// True for the settings the tile encoder serves: padded dim 64 or 128, 2 to 4
// bits per angle, padded_dim / 2 QJL rows.
inline bool tq_tile_ok(int padded_dim, int bits, int qjl_dim) {
  return (padded_dim == 64 || padded_dim == 128) && qjl_dim == padded_dim / 2 && bits >= 2 && bits <= 4;
}

// Launches the encoder; the caller checks launch_status.
void launch_tq_encode(const TqEncodeArgs& a, hipStream_t stream);

}  // namespace vrm
