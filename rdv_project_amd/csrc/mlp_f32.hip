// Exact-fp32 chain kernels: the reference's per-thread evaluation order on the
// fp32 matrix cores.
//
// The reference's order, per output:
//  - Linear (src/rdv/shaders/maps/linear.h:36-43):  acc = b[o]; acc += x[k] * W[o][k]
//  - LinearFast on a partial workgroup (linear_fast.h:102-108): the same fp32 loop
//  - LinearFast on a full workgroup (linear_fast.h:61-98) emulated exactly as
//    written: x and W rounded to fp16, products summed in fp32 from zero, then
//    the fp32 bias added.
// They serve chains containing an fp32 Linear layer, shapes without a matrix-core
// instantiation, and the < 32-row tail group that the reference evaluates in fp32.
//
// v_mfma_f32_16x16x4f32 computes D = C + A B as four chained fused multiply-adds
// in ascending k with one fp32 rounding each (every element of 200 random
// products equals fmaf(a3, b3, fmaf(a2, b2, fmaf(a1, b1, fmaf(a0, b0, c)))),
// denormals and infinities included), so feeding it k = 0..3, 4..7, ... IS the
// reference's loop, bit for bit.
#include <algorithm>
#include <cstddef>

#include "mlp_layout.h"
#include "rdv_common.h"

namespace rdv {

// One unit of work of staging parameters into LDS: 16-byte pieces, one per
// thread, of consecutive rows of a row-major fp32 matrix (a bias is one row).
struct ChainStageSlot {
  const float* src;  // first element of the slot's first row
  int dst;           // LDS float offset of that row
  int stride;        // LDS row stride in floats
  int iw;            // columns; past them kChainPad
  int units;         // pieces of this slot (<= threads per block)
  float inv_kq;      // 1 / pieces per row, pieces per row = ceil(iw / 4)
  int vec_f16;       // bit 0: rows of whole 16-byte pieces, 16-byte aligned; bit 1: round the values to fp16
};
constexpr int kChainSlots = 64;
constexpr int kChainStageBatch = 8;  // slots whose loads are all in flight before the first LDS write

// One layer's shape and places (32-bit words, read from LDS).
struct ChainLayer {
  int in_w, out_w, act;
  int f16;       // LinearFast emulation (fp16 operands, sum from zero, bias last)
  int woff;      // LDS float offset of the weights; < 0: read from W
  int wstride;   // LDS row stride in floats
  int boff;      // LDS float offset of the bias
  int reserved;
  const float* W;  // row-major fp32
};

struct ChainF32Args {
  const float* x;
  float* y;
  int64_t row0, nrows;  // rows handled by this launch: [row0, row0 + nrows)
  int64_t tiles;        // 16-row tiles
  int L, nslots;
  int encoding, enc_d, enc_l;
  int reserved;
  ChainLayer layer[RDV_MLP_MAX_LAYERS];
  ChainStageSlot slot[kChainSlots];
};
static_assert(sizeof(ChainF32Args) <= 4096 && sizeof(ChainF32Args) % 16 == 0, "kernel arguments");
constexpr int kChainHeadFloats = int(offsetof(ChainF32Args, slot) / 4);  // all but the slots
static_assert(kChainHeadFloats % 4 == 0, "the staged parameters start 16-byte aligned");

// A wave-uniform word of the argument block in LDS.
__device__ __forceinline__ int chain_u(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ const float* chain_u(const float* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  return reinterpret_cast<const float*>(uint64_t(uint32_t(chain_u(int(v)))) | uint64_t(uint32_t(chain_u(int(v >> 32)))) << 32);
}

// Feature of layer-0's input: raw, or the frequency encoding's f-th value.
__device__ __forceinline__ float chain_input(const ChainF32Args& a, const float* xr, int f) {
  const int D = a.enc_d;
  if (f < D) return xr[f];
  if (a.encoding != RDV_ENC_FREQ || f >= D * (1 + 2 * a.enc_l)) return 0.0f;
  const int k = (f - D) / (2 * D), r = (f - D) % (2 * D);
  const float t = ldexpf(xr[r < D ? r : r - D], k);  // 2^k p, exact
  return r < D ? sinpif(t) : cospif(t);
}

// What stands for a weight past a layer's last column: times the +0 its input is
// padded with it leaves every sum as it is, a sum of -0 too (+0 would make that +0).
constexpr float kChainPad = -0.0f;

// Weights W[row][16 c + 4 s + q], s = 0..3, of chunk c for this lane: from LDS
// (columns past the layer's width are staged as kChainPad up to a multiple of 4; the
// callers ask for no later ones), or from the layer's own rows.
template <bool LDSW>
__device__ __forceinline__ float chain_weight(const float* w, int row, int k, int iw, bool f16) {
  if constexpr (LDSW) {
    return w[row + k];
  } else {
    float v = w[row + (k < iw ? k : 0)];
    if (f16) v = float(half_t(v));
    return k < iw ? v : kChainPad;
  }
}

// A conditional body the compiler must branch around: matrix instructions have no
// side effects, and it would otherwise run every chunk unconditionally and
// select the results.
__device__ __forceinline__ void chain_branch() { asm volatile(""); }

// One layer for a wave's 16 rows: act[4 t + j] of lane (q, m) holds feature
// 16 t + 4 j + q of row m, in and out.  The A operand's row m' = 4 q' + j' of
// M tile t carries output 16 t + 4 j' + q', so D register j of lane (q, m) is
// output 16 t + 4 j + q: the B operand of the next layer's MFMA 4 t + j, whose
// k index q stands for feature 4 (4 t + j) + q.  Features stay in ascending k
// order through the chain with no lane exchange.
//
// M: tiles of 16 outputs.  KC > 0: the layer reads exactly KC chunks of 16
// inputs, straight-line (the next chunk's reads go out under this chunk's
// MFMAs); 0: any width, a branch per chunk.  FULL: exactly 16 M outputs, so no
// lane has a row or an output past the layer (the selects cost more vector-ALU
// time than a third of the MFMAs: the two add up on a SIMD).
template <int MT, int M, int KC, bool FULL, bool LDSW>
__device__ __forceinline__ void chain_layer_m(const ChainF32Args& a, int l, const float* sm, int lane,
                                              float (&act)[4 * MT]) {
  const ChainLayer& y = a.layer[l];
  // opaque, so that the lane's masks and addresses are formed per layer and not
  // hoisted out of the tile loop for every variant at once
  asm volatile("" : "+v"(lane));
  const int q = lane >> 4, m = lane & 15;
  const int fo = 4 * (m & 3) + (m >> 2);  // output (within its tile of 16) carried by A row m
  const int iw = chain_u(y.in_w), ow = chain_u(y.out_w), an = chain_u(y.act);
  const bool f16 = chain_u(y.f16) != 0;
  const int ki = KC > 0 ? 4 * KC : (iw + 3) >> 2;
  const float* sb = sm + chain_u(y.boff) + (FULL ? q : 0);
  const float* const w0 = LDSW ? sm + chain_u(y.woff) : chain_u(y.W);
  const int ws = LDSW ? chain_u(y.wstride) : iw;
  auto bias = [&](int i) { return sb[FULL ? 4 * i : (4 * i + q < ow ? 4 * i + q : 0)]; };
  f32x4 acc[M];
  int wr[M];  // this lane's row of each tile
#pragma unroll
  for (int t = 0; t < M; ++t) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[t][j] = bias(4 * t + j);
    const int o = FULL || 16 * t + fo < ow ? 16 * t + fo : ow - 1;  // a row past ow repeats the last; its outputs are zeroed
    wr[t] = o * ws;
  }
  if (f16) {
    chain_branch();
#pragma unroll
    for (int t = 0; t < M; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 4 * (KC > 0 ? KC : MT); ++i) act[i] = float(half_t(act[i]));
  }
#pragma unroll
  for (int c = 0; c < (KC > 0 ? KC : MT); ++c) {
    if (KC > 0 || 4 * c + 4 <= ki) {  // a whole chunk of 16 columns: 4 reads per tile, then 4 MFMAs on each tile's own chain
      int qc = q;
      if constexpr (KC == 0) {
        chain_branch();
        asm volatile("" : "+v"(qc));  // this chunk's addresses are formed here
      }
      constexpr int B = M <= 4 ? 4 : 1;  // steps whose weights are read together (registers)
#pragma unroll
      for (int s0 = 0; s0 < 4; s0 += B) {
        float w[M][B];
#pragma unroll
        for (int t = 0; t < M; ++t)
#pragma unroll
          for (int s = 0; s < B; ++s) w[t][s] = chain_weight<LDSW>(w0, wr[t], 16 * c + 4 * (s0 + s) + qc, iw, f16);
#pragma unroll
        for (int s = 0; s < B; ++s)
#pragma unroll
          for (int t = 0; t < M; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t][s], act[4 * c + s0 + s], acc[t], 0, 0, 0);
        if (B == 1) __builtin_amdgcn_sched_barrier(0);
      }
    } else if (4 * c < ki) {
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        if (4 * c + s < ki) {
          chain_branch();
          int qc = q;
          asm volatile("" : "+v"(qc));
#pragma unroll
          for (int t = 0; t < M; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(chain_weight<LDSW>(w0, wr[t], 16 * c + 4 * s + qc, iw, f16),
                                                          act[4 * c + s], acc[t], 0, 0, 0);
        }
      }
    }
  }
  if (f16) {
    chain_branch();
#pragma unroll
    for (int i = 0; i < 4 * M; ++i) acc[i / 4][i & 3] += bias(i);
  }
  if (an == RDV_ACT_RELU) {
    chain_branch();
#pragma unroll
    for (int i = 0; i < 4 * M; ++i) acc[i / 4][i & 3] = fmaxf(acc[i / 4][i & 3], 0.0f);
  }
#pragma unroll
  for (int i = 0; i < 4 * MT; ++i) {
    if (i / 4 < M) {
      const float v = acc[i / 4 < M ? i / 4 : 0][i & 3];
      act[i] = FULL || 4 * i + q < ow ? v : 0.0f;  // features past ow: zero times the next layer's zero columns
    } else {
      act[i] = 0.0f;
    }
  }
  if (an != RDV_ACT_RELU && an != RDV_ACT_NONE) {
    // one copy of the transcendental activations: a rolled loop over the features,
    // register i picked and replaced by selects
#pragma nounroll
    for (int i = 0; i < 4 * M; ++i) {
      float v = act[0];
#pragma unroll
      for (int k = 1; k < 4 * M; ++k) v = k == i ? act[k] : v;
      const int o = 4 * i + q;
      v = o < ow ? apply_act(an, o, v) : 0.0f;
#pragma unroll
      for (int k = 0; k < 4 * M; ++k) act[k] = k == i ? v : act[k];
    }
  }
}

template <int MT, bool LDSW>
__device__ __forceinline__ void chain_layer(const ChainF32Args& a, int l, const float* sm, int lane,
                                            float (&act)[4 * MT]) {
  const int ow = chain_u(a.layer[l].out_w), iw = chain_u(a.layer[l].in_w);
  const int mt = (ow + 15) >> 4;  // M tiles of 16 outputs
  if constexpr (MT == 4) {
    if constexpr (LDSW) {
      // square layers and heads of the common widths, straight-line
      if (iw == 64 && ow == 64) return chain_layer_m<MT, 4, 4, true, true>(a, l, sm, lane, act);
      if (iw <= 12 && ow == 64) return chain_layer_m<MT, 4, 0, true, true>(a, l, sm, lane, act);  // coordinates
      if (iw == 64 && mt == 1) return chain_layer_m<MT, 1, 4, false, true>(a, l, sm, lane, act);
      if (iw == 32 && ow == 32) return chain_layer_m<MT, 2, 2, true, true>(a, l, sm, lane, act);
    }
    switch (mt) {
      case 1: chain_layer_m<MT, 1, 0, false, LDSW>(a, l, sm, lane, act); break;
      case 2: chain_layer_m<MT, 2, 0, false, LDSW>(a, l, sm, lane, act); break;
      case 3: chain_layer_m<MT, 3, 0, false, LDSW>(a, l, sm, lane, act); break;
      default: chain_layer_m<MT, 4, 0, false, LDSW>(a, l, sm, lane, act); break;
    }
  } else {
    if (mt <= 4) chain_layer_m<MT, 4, 0, false, LDSW>(a, l, sm, lane, act);
    else if (mt <= 8) chain_layer_m<MT, 8, 0, false, LDSW>(a, l, sm, lane, act);
    else chain_layer_m<MT, 16, 0, false, LDSW>(a, l, sm, lane, act);
  }
}

// Persistent blocks; a block's waves take its 16-row tiles in turn, activations
// in registers throughout.  Parameters are staged into LDS once per block: rows
// at a stride of an odd number of 16-byte pieces, so that a wave's 16 rows x 4
// columns of a read fall into 64 different banks; every load of a batch of slots
// is in flight before the first write (one memory round trip per batch, not per
// layer), and the first tile's input rows before them.  A layer that does not
// fit is read from its own rows in global memory.
//
// Bound: the fp32 matrix rate (32 cycles per MFMA of 2,048 operations) plus the
// vector ALU's hand-off, which adds to it.  A coordinate network 3 -> 64 x 4 -> 4
// takes 212 MFMAs per 16 rows: 12.7 us for 65,536 rows on 1,024 SIMDs.  Measured,
// back to back: 24.8 us (3 us staging, 17 us of layers, start and end; 47.6-50 us
// for one row per lane on the vector ALUs with LDS broadcasts), 12.1 us for 8 rows
// (1.4 us per 64-wide layer of a single wave; 550 us for one thread per row).
// Tiles of 16 rather than 32 rows (v_mfma_f32_32x32x2f32, the same rate) spend
// half as much on the 4-wide head and the 3-wide input, and give small calls twice
// the waves.
template <int MT>
__device__ __forceinline__ void chain_f32_body(const ChainF32Args& ga, float* smem) {
  const int threads = int(blockDim.x), tid = int(threadIdx.x);
  // The layers' descriptions are copied to LDS by all threads at once and read
  // from there: indexed scalar loads would be a memory round trip per layer.
  using KernArg = const __attribute__((address_space(4))) uint8_t;
  KernArg* const ka = (KernArg*)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t* const ka32 = (const uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
  for (int i = tid; i < kChainHeadFloats; i += threads) reinterpret_cast<uint32_t*>(smem)[i] = ka32[i];
  const ChainF32Args& a = *reinterpret_cast<const ChainF32Args*>(smem);
  float* const sm = smem + kChainHeadFloats;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t per_block = (ga.tiles + gridDim.x - 1) / gridDim.x;
  const int64_t t_begin = int64_t(blockIdx.x) * per_block;
  const int64_t t_end = t_begin + per_block < ga.tiles ? t_begin + per_block : ga.tiles;
  const int D = ga.enc_d, in0 = ga.layer[0].in_w;
  // act[i] of lane (q, m): feature 4 i + q of row m of the tile; past in0 the row's
  // last one, zeroed by mask_raw (the wide kernel has no registers to put that off).
  // Loads only, four to a branch: a select beside each one waited for it, a memory
  // latency per four features of every tile (262,144 rows of 64 -> 64 -> 64 -> 16: 303 us,
  // now 61; 164 on the vector ALUs).
  auto load_raw = [&](int64_t tile, float (&act)[4 * MT]) {
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));  // per-tile masks and addresses, as in chain_layer_m
    const int q = lane >> 4;
    const int64_t r = tile * 16 + (lane & 15);
    const float* xr = ga.x + (ga.row0 + (r < ga.nrows ? r : ga.nrows - 1)) * D;
#pragma unroll
    for (int c = 0; c < MT; ++c) {
      if (16 * c < in0) {
        chain_branch();
#pragma unroll
        for (int i = 4 * c; i < 4 * c + 4; ++i) act[i] = xr[min(4 * i + q, in0 - 1)];
        if (MT > 4 && 16 * c + 16 > in0) {
#pragma unroll
          for (int i = 4 * c; i < 4 * c + 4; ++i) act[i] = 4 * i + q < in0 ? act[i] : 0.0f;
        }
      } else if (MT > 4) {
#pragma unroll
        for (int i = 4 * c; i < 4 * c + 4; ++i) act[i] = 0.0f;
      }
    }
  };
  auto mask_raw = [&](float (&act)[4 * MT]) {
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int q = lane >> 4;
#pragma unroll
    for (int c = 0; c < MT; ++c)
      if (16 * c + 16 > in0) {
        chain_branch();
#pragma unroll
        for (int i = 4 * c; i < 4 * c + 4; ++i) act[i] = 4 * i + q < in0 ? act[i] : 0.0f;
      }
  };
  const bool freq = ga.encoding == RDV_ENC_FREQ;
  float act[4 * MT] = {};
  // the first tile's rows are on their way while the parameters are staged
  if (!freq && t_begin + wave < t_end) load_raw(t_begin + wave, act);
  using KSlot = const __attribute__((address_space(4))) ChainStageSlot;
  KSlot* const slots = (KSlot*)(ka + offsetof(ChainF32Args, slot));
  const int nslots = ga.nslots;
#pragma nounroll
  for (int s0 = 0; s0 < nslots; s0 += kChainStageBatch) {  // the table is padded with copies of its last slot
    f32x4 v[kChainStageBatch];
    int dst[kChainStageBatch];
#pragma unroll
    for (int k = 0; k < kChainStageBatch; ++k) {
      KSlot& s = slots[s0 + k];
      const int u = min(tid, s.units - 1);               // spare threads repeat the last piece (same bytes)
      const int r = int((float(u) + 0.5f) * s.inv_kq);   // row, exact: u < 1024, at most 64 pieces per row
      const int c4 = 4 * (u - r * ((s.iw + 3) >> 2));    // first column
      const float* const src = s.src;
      dst[k] = s.dst + r * s.stride + c4;
      if (s.vec_f16 & 1) {
        v[k] = reinterpret_cast<const f32x4*>(src)[u];
      } else {
        const int e = r * s.iw + c4, last = s.iw - 1 - c4;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[k][j] = src[e + min(j, last)];
#pragma unroll
        for (int j = 1; j < 4; ++j) v[k][j] = j <= last ? v[k][j] : kChainPad;
      }
    }
#pragma unroll
    for (int k = 0; k < kChainStageBatch; ++k) {
      if (slots[s0 + k].vec_f16 & 2) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[k][j] = float(half_t(v[k][j]));
      }
      *reinterpret_cast<f32x4*>(sm + dst[k]) = v[k];
    }
  }
  __syncthreads();

  const int L = chain_u(a.L), ow = chain_u(a.layer[L - 1].out_w);
  for (int64_t tile = t_begin + wave; tile < t_end;) {
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    const int q = lane >> 4;
    const int64_t r = tile * 16 + (lane & 15);
    if (freq) {
      const float* xr = ga.x + (ga.row0 + (r < ga.nrows ? r : ga.nrows - 1)) * D;
#pragma unroll
      for (int i = 0; i < 4 * MT; ++i) act[i] = 0.0f;
#pragma nounroll
      for (int i = 0; 4 * i < in0; ++i) {  // one copy of sinpi / cospi, as for the activations
        const float v = 4 * i + q < in0 ? chain_input(ga, xr, 4 * i + q) : 0.0f;
#pragma unroll
        for (int k = 0; k < 4 * MT; ++k) act[k] = k == i ? v : act[k];
      }
    } else if (MT == 4) {
      mask_raw(act);
    }
#pragma nounroll
    for (int l = 0; l < L; ++l) {
      if (chain_u(a.layer[l].woff) >= 0) chain_layer<MT, true>(a, l, sm, lane, act);
      else chain_layer<MT, false>(a, l, sm, lane, act);
    }
    if (r < ga.nrows) {
      float* yr = ga.y + (ga.row0 + r) * ow;
#pragma unroll
      for (int i = 0; i < 4 * MT; ++i)
        if (4 * i < ow) {
          chain_branch();
          if (4 * i + q < ow) yr[4 * i + q] = act[i];
        }
    }
    tile += threads >> 6;
    if (!freq && tile < t_end) load_raw(tile, act);
  }
}

// Widths up to 64 (16 + 16 registers of activations and sums: four waves per SIMD).
__global__ __launch_bounds__(1024) void mlp_chain_f32_reg_kernel(ChainF32Args ga) {
  extern __shared__ __attribute__((aligned(16))) float smem_f32[];
  chain_f32_body<4>(ga, smem_f32);
}

// Widths up to 256.
__global__ __launch_bounds__(512) void mlp_chain_f32_kernel(ChainF32Args ga) {
  extern __shared__ __attribute__((aligned(16))) float smem_f32[];
  chain_f32_body<16>(ga, smem_f32);
}

constexpr int kChainNarrow = 64;                   // widest layer of mlp_chain_f32_reg_kernel
constexpr int64_t kChainLdsFloats = 156 * 1024 / 4;  // parameters staged in LDS (160 KiB per block)

static bool chain_narrow(const MlpLayout& lay) {
  for (int l = 0; l < lay.n_layers; ++l)
    if (lay.in_w[l] > kChainNarrow || lay.out_w[l] > kChainNarrow) return false;
  return true;
}

// The kernel that evaluates the chain in exact fp32.
const char* chain_f32_name(const MlpLayout& lay) {
  return chain_narrow(lay) ? "mlp_chain_f32_reg_kernel" : "mlp_chain_f32_kernel";
}

int launch_mlp_chain_f32(const rdv_mlp_desc& d, const MlpLayout& lay, const void* packed, const float* x, float* y,
                         int64_t row0, int64_t nrows, bool force_f32, hipStream_t stream, const DirectWeights* dw) {
  if (nrows <= 0) return RDV_OK;
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc != RDV_OK) return rc;
  const bool narrow = chain_narrow(lay);
  ChainF32Args a = {};
  a.x = x;
  a.y = y;
  a.row0 = row0;
  a.nrows = nrows;
  a.tiles = (nrows + 15) / 16;
  a.L = d.n_layers;
  a.encoding = d.encoding;
  a.enc_d = d.in_features;
  a.enc_l = d.enc_octaves;
  // One block per CU, spread over as many CUs as there are groups of 4 tiles (a
  // wave on each SIMD).  Past 8 tiles per CU the narrow kernel takes 16 waves:
  // their LDS reads hide behind each other's MFMAs (65,536 rows of the 64-wide
  // chain: 24.8 us, 27.7 with 8 waves of two tiles each).
  const int64_t blocks = std::min<int64_t>(di.cu_count, (a.tiles + 3) / 4);
  const int threads = narrow && a.tiles > 8 * blocks ? 1024 : 512;
  const uint8_t* pk = static_cast<const uint8_t*>(packed);
  const int64_t cap = std::min<int64_t>(kChainLdsFloats, int64_t(di.lds_per_block) / 4) - kChainHeadFloats;
  int off = 0;
  auto stage = [&](const float* src, int rows, int iw, int stride, int f16) {
    const int kq = (iw + 3) / 4;
    const int vec = iw % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0 ? 1 : 0;
    const int per = threads / kq;  // rows per slot
    for (int r = 0; r < rows; r += per) {
      const int n = std::min(per, rows - r);
      a.slot[a.nslots++] = {src + int64_t(r) * iw, off + r * stride, stride, iw, n * kq, 1.0f / float(kq), vec | 2 * f16};
    }
    off += rows * stride;
  };
  for (int l = 0; l < a.L; ++l) {
    const int iw = lay.in_w[l], ow = lay.out_w[l];
    ChainLayer& y = a.layer[l];
    y.W = dw != nullptr ? dw->W[l] : reinterpret_cast<const float*>(pk + lay.w32_off[l]);
    y.in_w = iw;
    y.out_w = ow;
    y.act = d.act[l];
    y.f16 = (d.prec[l] == RDV_PREC_F16 && !force_f32) ? 1 : 0;
    y.boff = off;
    stage(dw != nullptr ? dw->b[l] : reinterpret_cast<const float*>(pk + lay.b32_off[l]), 1, ow, (ow + 3) & ~3, 0);
  }
  for (int l = 0; l < a.L; ++l) {
    const int kq = (lay.in_w[l] + 3) / 4;
    const int stride = 4 * (kq | 1);  // an odd number of 16-byte pieces
    const int per = threads / kq;
    const int slots = (lay.out_w[l] + per - 1) / per;
    ChainLayer& y = a.layer[l];
    y.wstride = stride;
    if (off + int64_t(lay.out_w[l]) * stride > cap || a.nslots + slots > kChainSlots - kChainStageBatch) {
      y.woff = -1;
      continue;
    }
    y.woff = off;
    stage(y.W, lay.out_w[l], lay.in_w[l], stride, y.f16);
  }
  for (int k = 0; k < kChainStageBatch; ++k) a.slot[a.nslots + k] = a.slot[a.nslots - 1];
  const void* fn = narrow ? reinterpret_cast<const void*>(&mlp_chain_f32_reg_kernel)
                          : reinterpret_cast<const void*>(&mlp_chain_f32_kernel);
  static bool raised[2] = {};
  if (!raised[narrow]) {
    RDV_HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(std::min<int64_t>(kChainLdsFloats * 4, int64_t(di.lds_per_block)))));
    raised[narrow] = true;
  }
  void* params[] = {&a};
  RDV_HIP_TRY(hipLaunchKernel(fn, dim3(unsigned(blocks)), dim3(unsigned(threads)), params, size_t(kChainHeadFloats + off) * 4, stream));
  return RDV_OK;
}

}  // namespace rdv
