// Pieces shared by the training kernels (train.hip, train_fused.hip): the
// tile-fragment feature order, the selection fragments that turn a fragment's
// lanes from points to features, and sums over a wave.
#ifndef RDV_TRAIN_TILE_H
#define RDV_TRAIN_TILE_H

#include "mlp_core.h"

namespace rdv {

// Sum over a wave (every lane gets it): DPP row shifts + row broadcasts.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float tr_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, true));
}
__device__ __forceinline__ float tr_wave_sum(float v) {
  v += tr_dpp<0x111, 0xF>(v);
  v += tr_dpp<0x112, 0xF>(v);
  v += tr_dpp<0x114, 0xF>(v);
  v += tr_dpp<0x118, 0xF>(v);
  v += tr_dpp<0x142, 0xA>(v);
  v += tr_dpp<0x143, 0xC>(v);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

typedef half_t half4v __attribute__((ext_vector_type(4)));

// Tile-fragment layout of the step's intermediate fp16 buffers (the kept hidden
// activations h_i, the head gradient g and the gradients g_i between backward
// launches), [rows][W] with rows a multiple of 64: 32-point tiles of
// Wp = 16 ceil(W / 16) features, tile k at k 32 Wp; within a tile, 16-byte chunk
// c = 64 s + 32 hh + col holds point col, features 16 s + 4 hh + 0..3 and then
// 16 s + 8 + 4 hh + 0..3 (tfl_feature).  That chunk is lane 32 hh + col's B
// fragment of K chunk s in the hidden (chunk_sigma) order, and equally the fp16
// of D registers 8 (s % 2) .. + 7 of 32-row block s / 2, so a wave writes or
// reads a whole 1 KiB slot s with one 16-byte access per lane.  Features past W
// are stored as zeros.
__device__ __forceinline__ int tfl_feature(int s, int hh, int j) { return 16 * s + 4 * hh + (j & 3) + ((j >> 2) << 3); }

// 0/1 fragment par: lane (n = lane % 32, hh = lane / 32), element j is 1 where
// tfl_feature(par, hh, j) == n.  A x select(0) + A' x select(1) turns the K
// slots of two consecutive 16-feature chunks (or of the two 16-point halves of
// a K = points fragment pair) into the 32 columns of D.
__device__ __forceinline__ half8 tp2_select(int par, int lane) {
  half8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = tfl_feature(par, lane >> 5, j) == (lane & 31) ? half_t(1.0f) : half_t(0.0f);
  return v;
}

// D registers 8 ks .. 8 ks + 7 as fp16 (points tfl_feature(ks, h, 0..7) of a
// point-major product; features 32 block + tfl_feature(ks, h, 0..7) of a
// feature-major one).
__device__ __forceinline__ half8 tp2_half(const f32x16& d, int ks) {
  half8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = half_t(d[8 * ks + j]);
  return v;
}

// Sum of 8 fp16 values into an fp32 accumulator.
__device__ __forceinline__ float tp2_sum(const half8& v, float acc) {
#pragma unroll
  for (int j = 0; j < 8; j += 2) acc = __builtin_amdgcn_fdot2(half2v{v[j], v[j + 1]}, half2v{1, 1}, acc, false);
  return acc;
}

// 0/1 fragment for the natural feature order of chunk par: lane (n, hh),
// element j is 1 where 16 par + 8 hh + j == n.
__device__ __forceinline__ half8 tp2_select_nat(int par, int lane) {
  half8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = 16 * par + 8 * (lane >> 5) + j == (lane & 31) ? half_t(1.0f) : half_t(0.0f);
  return v;
}

}  // namespace rdv

#endif  // RDV_TRAIN_TILE_H
