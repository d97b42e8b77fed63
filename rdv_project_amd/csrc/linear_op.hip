// Per-layer tensor operations: y[rows, out] = x[rows, in] W^T + b and
// y = max(x, 0), one dispatch per op, fp32 buffers in and out.
//
// Reference: the TensorOperation family (src/rdv/maths/__init__.py:1251-1380),
//   LinearTensorOp       src/rdv/shaders/tensors/linear_tensor_op.h:8-51       (fp32)
//   LinearTensorOpSmall  src/rdv/shaders/tensors/linear_tensor_op_small.h:50-247 (fp16 x, W; fp32 acc)
//   LinearTensorOpSimple src/rdv/shaders/tensors/linear_tensor_op_simple.h:49-116
//   LinearTensorOpFast   src/rdv/shaders/tensors/linear_tensor_op_fast.h:37-122
//   LinearTensorOpMine   src/rdv/shaders/tensors/linear_tensor_op_mine.h:51-133
//   ReLUTensorOp         src/rdv/shaders/tensors/relu_tensor_op.h:3-22
// The four fp16 variants compute the same function (x and W rounded to fp16,
// products accumulated in fp32, fp32 bias) and differ only in tiling, so one
// kernel serves them; the weight may arrive as fp32 [out, in] (read and rounded
// at dispatch, like Small and Mine), fp16 [out, in] (Simple's pre-cast copy) or
// fp16 [out/16][in/16][16 k][16 n] tiles (Fast's pre-tiled copy, nn.py:472-490).
//
// linear_gemm_kernel (below) serves most shapes, linear_stream_kernel large products
// over few columns; relu_op_kernel streams.
#include <algorithm>

#include "rdv_common.h"

namespace rdv {

namespace {

__device__ __forceinline__ half8 to_half8(f32x4 a, f32x4 b) {
  half8 h;
  h[0] = half_t(a[0]); h[1] = half_t(a[1]); h[2] = half_t(a[2]); h[3] = half_t(a[3]);
  h[4] = half_t(b[0]); h[5] = half_t(b[1]); h[6] = half_t(b[2]); h[7] = half_t(b[3]);
  return h;
}

// ---------------------------------------------------------------- linear ops
// A tiled product.  A block of NW waves (2 across the rows, NW / 2 across the
// outputs) computes BM rows x BN outputs; per K step of 64 (fp16) or 32 (fp32)
// columns it stages both operands' tiles in LDS as MFMA fragments, double
// buffered: the next step's global loads are in flight during this step's MFMAs,
// and one barrier per step suffices.  D^T = W x^T, so a lane ends with 4
// consecutive outputs of one row: one cached 16-byte store per 16 x 16 tile.
//   fp16: v_mfma_f32_16x16x32_f16 over chunks of 32 columns, x rounded on the way
//         into LDS; fp32: v_mfma_f32_16x16x4f32 over chunks of 16 (quarter q holds
//         columns 4q + s in step s).  Bias first, chunks ascending.
// TILED: the weight is the fp16 tile layout [out/16][in/16][16 k][16 n].  Its
// tiles go from global memory straight into LDS (global_load_lds_dwordx4) and
// the fragments' transpose is done by ds_read_b64_tr_b16, which hands lane i of 16
// column i of a 4 x 16 block (through registers it is eight 2-byte loads per piece).
// Pieces staged through registers are written at lane position
// 16 q + (r + 2 (q + 4 c)) % 16 for (row r, quarter q, chunk c): the 8 lanes that
// hold one row's 8 pieces write 8 different 16-byte bank groups, and a read is
// still one permuted 1 KiB run.
//
// Bound: HBM for narrow layers (524,288 x 128 -> 128: 112 us, 4.8 TB/s, a copy's
// rate); for wide ones the tiles' stores: a chip's tiles run in step, so every CU
// writes its 256 KiB at once and computes nothing meanwhile (65,536 x 1024 -> 1024
// fp16: 141 us of 199 without the stores).  Measured against restaging the weight
// per 64 rows and 256 columns: that shape 1055 -> 199 us, 65,536 x 512 -> 512 fp32
// 642 -> 280 us (123 TFLOP/s).
__device__ __attribute__((aligned(16))) uint32_t g_lg_zero16[4] = {0u, 0u, 0u, 0u};
typedef __fp16 lg_half4 __attribute__((ext_vector_type(4)));

struct LinearGemmArgs {
  const float* x;
  const void* w;
  const float* bias;
  float* y;
  int64_t rows, row_tiles;
  int64_t block0;  // this launch's first block
  int in, out, col_tiles;
  int wkind, relu;
};

// 16 bytes per lane from src to LDS byte address lds_wave + 16 lane (below 64 KiB).
__device__ __forceinline__ void lg_dma16(const void* src, uint32_t lds_wave) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(src), "s"(__builtin_amdgcn_readfirstlane(lds_wave))
      : "memory");
}

template <int NW, int WM, int WN>
struct LgLds {
  static constexpr int kX = 2 * WM * 2 * 1024, kW = NW / 2 * WN * 2 * 1024;  // bytes per buffer
  static constexpr int kBytes = 2 * (kX + kW);
};

template <bool F16, bool TILED, int NW, int WM, int WN>
__global__ __launch_bounds__(64 * NW, 2) void linear_gemm_kernel(LinearGemmArgs a) {
  using LD = LgLds<NW, WM, WN>;
  constexpr int NN = NW / 2;           // waves across the outputs (two across the rows)
  constexpr int BM = 32 * WM, BN = 16 * NN * WN;
  constexpr int NX = WM * 4 / NW;      // row pieces per thread and step (WN weight pieces)
  constexpr int PR = 8 * NW;           // rows between a thread's pieces
  constexpr int KS = F16 ? 64 : 32;    // columns per step, two chunks
  constexpr int PK = KS / 8;           // columns per 16-byte fragment piece
  constexpr bool kLate = F16 && !TILED && NW * WN == 32 && WM == 8;  // no registers for two chunks' weight fragments
  static_assert(!TILED || 2 * LD::kW <= 64 * 1024, "DMA targets below 64 KiB");
  extern __shared__ f32x4 lo_smem[];
  uint8_t* const sw = reinterpret_cast<uint8_t*>(lo_smem);  // W buffers first
  uint8_t* const sx = sw + 2 * LD::kW;
  const int tid = int(threadIdx.x), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / NN, wn = wave % NN;
  const int r = lane & 15, q = lane >> 4;
  // Blocks of one XCD (consecutive multiples of 8) take the column tiles of a
  // row tile one after the other, so its x rows are read from HBM once.
  const int64_t b = a.block0 + blockIdx.x;
  const int ct = int((b >> 3) % a.col_tiles);
  const int64_t rt = ((b >> 3) / a.col_tiles) * 8 + (b & 7);
  if (rt >= a.row_tiles) return;
  const int64_t row0 = rt * BM;
  const int o0 = ct * BN;
  const int in = a.in;

  // register-staged pieces: rows tid / 8 + PR i of the tile, piece tid % 8 of the step
  const int pr = tid >> 3, pp = tid & 7;
  const int spos = ((pp >> 2) * 64 + 16 * (pp & 3) + ((pr + 2 * pp) & 15)) * 16 + (pr >> 4) * 2048;
  const float* const xb = a.x + row0 * in;
  const int xlast = int(a.rows - row0 < BM ? a.rows - row0 : BM) - 1;
  const int olast = (a.out - o0 < BN ? a.out - o0 : BN) - 1;
  f32x4 xr[NX][F16 ? 2 : 1];
  f32x4 wr[TILED ? 1 : WN][F16 ? 2 : 1];

  auto load = [&](int k0, int buf) {
    const bool ok = k0 + pp * PK < in;  // a piece past `in` re-reads the step's first one and is zeroed when parked
    const int kk = k0 + (ok ? pp * PK : 0);
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int rr = min(pr + PR * i, xlast);
#pragma unroll
      for (int v = 0; v < (F16 ? 2 : 1); ++v) xr[i][v] = reinterpret_cast<const f32x4*>(xb + int64_t(rr) * in + kk)[v];
    }
    if constexpr (TILED) {
      // BN outputs x 4 k tiles of 512 bytes; a wave's instruction moves two neighbouring k tiles
#pragma unroll
      for (int i = 0; i < WN; ++i) {
        const int u = NW * i + wave;            // 1 KiB unit: output tile u / 2, k tiles 2 (u % 2), + 1
        const int ot = min(u >> 1, olast >> 4);
        const int kt = (k0 >> 4) + 2 * (u & 1) + (lane >> 5);
        const int piece = (lane & 31) ^ ((lane & 16) >> 1);  // rows 12..15 of a tile before rows 8..11
        const half_t* src = static_cast<const half_t*>(a.w) + (int64_t((o0 >> 4) + ot) * (in >> 4) + kt) * 256 + 8 * piece;
        lg_dma16(16 * kt < in ? static_cast<const void*>(src) : g_lg_zero16,
                 uint32_t(reinterpret_cast<uintptr_t>(sw + buf * LD::kW + u * 1024)));
      }
    } else {
#pragma unroll
      for (int i = 0; i < WN; ++i) {
        const int o = o0 + min(pr + PR * i, olast);
        const int64_t e = int64_t(o) * in + kk;
        if (F16 && a.wkind == RDV_WKIND_F16_TILED16) {  // a tile copy that is not 16-byte aligned
          const half_t* wt = static_cast<const half_t*>(a.w) + (int64_t(o >> 4) * (in >> 4) + (kk >> 4)) * 256 + (o & 15);
          half8 h;
#pragma unroll
          for (int j = 0; j < 8; ++j) h[j] = wt[((kk & 15) + j) * 16];
          wr[i][0] = __builtin_bit_cast(f32x4, h);
        } else if (F16 && a.wkind == RDV_WKIND_F16) {
          wr[i][0] = *reinterpret_cast<const f32x4*>(static_cast<const half_t*>(a.w) + e);
        } else {
#pragma unroll
          for (int v = 0; v < (F16 ? 2 : 1); ++v)
            wr[i][v] = reinterpret_cast<const f32x4*>(static_cast<const float*>(a.w) + e)[v];
        }
      }
    }
  };
  auto park = [&](int k0, int buf) {
    const bool ok = k0 + pp * PK < in;
    const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      f32x4 v;
      if constexpr (F16) v = __builtin_bit_cast(f32x4, to_half8(xr[i][0], xr[i][1]));
      else v = xr[i][0];
      *reinterpret_cast<f32x4*>(sx + buf * LD::kX + spos + i * (NN * 2048)) = ok ? v : zero4;
    }
    if constexpr (!TILED) {
#pragma unroll
      for (int i = 0; i < WN; ++i) {
        f32x4 v = wr[i][0];
        if constexpr (F16) {
          if (a.wkind == RDV_WKIND_F32) v = __builtin_bit_cast(f32x4, to_half8(wr[i][0], wr[i][1]));
        }
        *reinterpret_cast<f32x4*>(sw + buf * LD::kW + spos + i * (NN * 2048)) = ok ? v : zero4;
      }
    }
  };

  f32x4 acc[WM][WN];
#pragma unroll
  for (int n = 0; n < WN; ++n) {
    const int col = o0 + 16 * (WN * wn + n) + 4 * q;
    f32x4 bv;
#pragma unroll
    for (int j = 0; j < 4; ++j) bv[j] = a.bias[min(col + j, a.out - 1)];
#pragma unroll
    for (int m = 0; m < WM; ++m) acc[m][n] = bv;
  }
  load(0, 0);
  park(0, 0);
  if constexpr (TILED) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const int steps = (in + KS - 1) / KS;
  for (int s = 0; s < steps; ++s) {
    const bool more = s + 1 < steps;
    if (more) load((s + 1) * KS, (s + 1) & 1);
    const uint8_t* bx = sx + (s & 1) * LD::kX + wm * WM * 2048;
    const uint8_t* bw = sw + (s & 1) * LD::kW + wn * WN * 2048;
    // TILED, quarter q: rows 8 (q % 2) .. + 7 of k tile 2 c + q / 2, four at a time; odd
    // quarters find theirs swapped, so neighbouring quarters read different banks
    const uint32_t tlo = uint32_t(reinterpret_cast<uintptr_t>(bw)) + (q >> 1) * 512 + (q & 1) * 384 + r * 8;
    const uint32_t thi = uint32_t(reinterpret_cast<uintptr_t>(bw)) + (q >> 1) * 512 + (q & 1) * 256 + 128 - (q & 1) * 128 + r * 8;
    auto read_w = [&](int c, f32x4 (&wf)[WN]) {
      const int rpos = (c * 64 + 16 * q + ((r + 2 * (q + 4 * c)) & 15)) * 16;
#pragma unroll
      for (int n = 0; n < WN; ++n) {
        if constexpr (TILED) {
          typedef __attribute__((address_space(3))) lg_half4 lds_h4;
          const lg_half4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4*)(tlo + n * 2048 + c * 1024));
          const lg_half4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4*)(thi + n * 2048 + c * 1024));
          const f32x2 l2 = __builtin_bit_cast(f32x2, lo), h2 = __builtin_bit_cast(f32x2, hi);
          wf[n] = f32x4{l2[0], l2[1], h2[0], h2[1]};
        } else {
          wf[n] = *reinterpret_cast<const f32x4*>(bw + n * 2048 + rpos);
        }
      }
    };
    auto read_x = [&](int c, int m) {
      const int rpos = (c * 64 + 16 * q + ((r + 2 * (q + 4 * c)) & 15)) * 16;
      return *reinterpret_cast<const f32x4*>(bx + m * 2048 + rpos);
    };
    auto products = [&](int m, const f32x4 (&wf)[WN], const f32x4& xv) {
#pragma unroll
      for (int n = 0; n < WN; ++n) {
        if constexpr (F16) {
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wf[n]),
                                                             __builtin_bit_cast(half8, xv), acc[m][n], 0, 0, 0);
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k)
            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[n][k], xv[k], acc[m][n], 0, 0, 0);
        }
      }
    };
    constexpr int WB = kLate ? 1 : 2;
    // Both chunks' weight fragments and the first one's x fragments are on their way
    // before the first product; a row tile's second x fragment is read into the
    // first one's registers once its products are issued, so the reads of chunk 1
    // run under the products of chunk 0 (against reading each chunk before its
    // products: fp32 65,536 x 512 -> 512 287 -> 280 us, 18,624 x 512 -> 512 103 -> 98,
    // fp16 the same).
    f32x4 wf[WB][WN], xf[WM];
    read_w(0, wf[0]);
#pragma unroll
    for (int m = 0; m < WM; ++m) xf[m] = read_x(0, m);
    if constexpr (!kLate) read_w(1, wf[1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < WM; ++m) {
      products(m, wf[0], xf[m]);
      xf[m] = read_x(1, m);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kLate) read_w(1, wf[0]);
#pragma unroll
    for (int m = 0; m < WM; ++m) products(m, wf[WB - 1], xf[m]);
    __builtin_amdgcn_sched_barrier(0);
    if (more) park((s + 1) * KS, (s + 1) & 1);
    if constexpr (TILED) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

#pragma unroll
  for (int m = 0; m < WM; ++m) {
    const int64_t row = row0 + 16 * (WM * wm + m) + r;
    if (row < a.rows) {
      float* yr = a.y + row * a.out;
#pragma unroll
      for (int n = 0; n < WN; ++n) {
        const int col = o0 + 16 * (WN * wn + n) + 4 * q;
        if (col < a.out) {
          f32x4 v = acc[m][n];
          if (a.relu) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = fmaxf(v[j], 0.0f);
          }
          *reinterpret_cast<f32x4*>(yr + col) = v;
        }
      }
    }
  }
}

template <bool F16, bool TILED, int NW, int WM, int WN>
int launch_linear_gemm_t(const LinearGemmArgs& a0, hipStream_t stream) {
  constexpr int kBytes = LgLds<NW, WM, WN>::kBytes, BM = 32 * WM, BN = 8 * NW * WN;
  LinearGemmArgs a = a0;
  a.row_tiles = (a.rows + BM - 1) / BM;
  a.col_tiles = (a.out + BN - 1) / BN;
  const int64_t grid = (a.row_tiles + 7) / 8 * 8 * a.col_tiles;
  static bool attr = false;
  if (!attr) {
    RDV_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&linear_gemm_kernel<F16, TILED, NW, WM, WN>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kBytes));
    attr = true;
  }
  // A launch takes at most 2^32 - 1 threads (HIP keeps their count in 32 bits and runs
  // what is left of a larger one without an error): 1.07e9 rows of the smallest tile.
  constexpr int64_t kMaxBlocks = 0xffffffffLL / (64 * NW) / 8 * 8;  // whole XCD rounds
  for (a.block0 = 0; a.block0 < grid; a.block0 += kMaxBlocks) {
    const int64_t blocks = std::min(grid - a.block0, kMaxBlocks);
    linear_gemm_kernel<F16, TILED, NW, WM, WN><<<dim3(unsigned(blocks)), dim3(64 * NW), kBytes, stream>>>(a);
    RDV_HIP_TRY(hipGetLastError());
  }
  return RDV_OK;
}

// --------------------------------------------------------- few columns, many rows
// A persistent block of 4 waves owns up to 128 outputs: it stages their weights and
// biases in LDS once, as A fragments (slot (t, c, lane): W[o0 + 16 t + lane % 16][16 c +
// 4 (lane / 16) ..] for v_mfma_f32_16x16x4f32, [32 c + 8 (lane / 16) ..] for
// v_mfma_f32_16x16x32_f16), then its waves walk 32-row tiles
// with a grid stride and no barrier, the next tile's x loaded (16 bytes a lane)
// while this one is computed.  The products and their order are linear_gemm_kernel's.
//
// linear_gemm_kernel stages whole steps of 32 (fp16: 64) columns and its blocks load, compute and
// store in turn; with one or two steps there is little to overlap, and up to half of
// it is padding.  Bound: HBM.  Measured, gemm and this kernel: 262,144 x 8 -> 128 37.7 and
// 24.7 us, 65,536 x 48 -> 512 56 and 42, 65,536 x 16 -> 1024 76 and 47, 4,194,304 x 8 -> 4 111
// and 58; fp16 65,536 x 16 -> 1024 60 and 48, 4,194,304 x 8 -> 16 124 and 78.
constexpr int kLsThreads = 256, kLsWaves = 4, kLsOutputs = 128, kLsRows = 32;  // rows per wave and tile

struct LinearStreamArgs {
  const float* x;
  const void* w;
  const float* bias;
  float* y;
  int64_t rows, tasks;  // tasks: tiles of kLsWaves * kLsRows rows
  int in, out, wkind, relu;
  int ob, n_ob;         // outputs per block (a multiple of 16), blocks of outputs
};

template <bool F16, int NKC, int G>  // chunks of 32 (fp16) or 16 columns, tiles of 16 outputs stored together
__global__ __launch_bounds__(kLsThreads) void linear_stream_kernel(LinearStreamArgs a) {
  constexpr int KC = F16 ? 32 : 16, PV = F16 ? 2 : 1;  // columns per chunk, 16-byte loads per lane and chunk
  extern __shared__ f32x4 lo_smem[];
  const int nt = a.ob / 16;
  f32x4* const sw = lo_smem;                     // [nt][NKC][64]
  f32x4* const sb = lo_smem + nt * NKC * 64;     // [ob / 4]
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // blocks of the same rows are neighbours, so their x re-reads hit the shared cache
  const int o0 = int(blockIdx.x % unsigned(a.n_ob)) * a.ob;
  const int64_t stride = gridDim.x / unsigned(a.n_ob);
  const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = threadIdx.x; s < nt * NKC * 64; s += kLsThreads) {
    const int o = o0 + 16 * (s / (NKC * 64)) + (s & 15);
    const int k = KC * ((s >> 6) % NKC) + KC / 4 * ((s & 63) >> 4);
    f32x4 v = zero4;
    if (o < a.out && k < a.in) {
      const int64_t e = int64_t(o) * a.in + k;
      if (!F16) {
        v = *reinterpret_cast<const f32x4*>(static_cast<const float*>(a.w) + e);
      } else if (a.wkind == RDV_WKIND_F32) {
        const f32x4* src = reinterpret_cast<const f32x4*>(static_cast<const float*>(a.w) + e);
        v = __builtin_bit_cast(f32x4, to_half8(src[0], src[1]));
      } else {
        v = *reinterpret_cast<const f32x4*>(static_cast<const half_t*>(a.w) + e);
      }
    }
    sw[s] = v;
  }
  for (int i = threadIdx.x; i < a.ob; i += kLsThreads) reinterpret_cast<float*>(sb)[i] = o0 + i < a.out ? a.bias[o0 + i] : 0.0f;
  __syncthreads();

  f32x4 raw[2][NKC][PV], xf[2][NKC];
  // rows clamped into range (their results are not stored), columns past `in` to
  // column 0 (zeroed on use): every load is in bounds
  auto load = [&](int64_t task) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t row = (task * kLsWaves + wave) * kLsRows + 16 * h + r;
      const float* xr = a.x + (row < a.rows ? row : a.rows - 1) * a.in;
#pragma unroll
      for (int c = 0; c < NKC; ++c) {
        const int k = KC * c + KC / 4 * q;
#pragma unroll
        for (int v = 0; v < PV; ++v) raw[h][c][v] = reinterpret_cast<const f32x4*>(xr + (k < a.in ? k : 0))[v];
      }
    }
  };
  int64_t task = blockIdx.x / unsigned(a.n_ob);
  if (task < a.tasks) load(task);
  for (; task < a.tasks; task += stride) {
#pragma unroll
    for (int c = 0; c < NKC; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4 v = raw[h][c][0];
        if constexpr (F16) v = __builtin_bit_cast(f32x4, to_half8(raw[h][c][0], raw[h][c][PV - 1]));
        xf[h][c] = KC * c + KC / 4 * q < a.in ? v : zero4;
      }
    load(task + stride < a.tasks ? task + stride : a.tasks - 1);
    const int64_t row0 = (task * kLsWaves + wave) * kLsRows + r;
    float* const y0 = a.y + row0 * a.out + o0 + 4 * q;
    // G tiles of 16 outputs at a time, their stores together: 2 make whole 128-byte lines
    // of y; for a y past the caches 8, whole rows of the block (1,048,576 x 48 -> 256 404 us
    // with 2, 367 with 8; 65,536 x 48 -> 512 42.1 and 43.4).
    for (int t0 = 0; t0 < nt; t0 += G) {
      f32x4 acc[G][2];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int t = t0 + u < nt ? t0 + u : nt - 1;
        acc[u][0] = acc[u][1] = sb[4 * t + q];
#pragma unroll
        for (int c = 0; c < NKC; ++c) {
          const f32x4 wv = sw[(t * NKC + c) * 64 + lane];
          if constexpr (F16) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
              acc[u][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wv), __builtin_bit_cast(half8, xf[h][c]),
                                                                 acc[u][h], 0, 0, 0);
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
              for (int h = 0; h < 2; ++h) acc[u][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[k], xf[h][c][k], acc[u][h], 0, 0, 0);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (row0 + 16 * h < a.rows) {
#pragma unroll
          for (int u = 0; u < G; ++u) {
            if (t0 + u < nt && o0 + 16 * (t0 + u) + 4 * q < a.out) {
              if (a.relu) {
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[u][h][j] = fmaxf(acc[u][h][j], 0.0f);
              }
              *reinterpret_cast<f32x4*>(y0 + int64_t(16 * h) * a.out + 16 * (t0 + u)) = acc[u][h];
            }
          }
        }
      }
    }
  }
}

template <bool F16, int NKC, int G>
int launch_linear_stream_t(const LinearStreamArgs& a, int cu, hipStream_t stream) {
  const size_t lds = size_t(a.ob / 16) * NKC * 1024 + size_t(a.ob) * 4;  // at most 32.5 KiB
  int occ = 0;
  RDV_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, linear_stream_kernel<F16, NKC, G>, kLsThreads, lds));
  const int64_t slots = int64_t(cu) * std::max(occ, 1);
  const int64_t groups = std::max<int64_t>(1, std::min<int64_t>(a.tasks, (slots + a.n_ob - 1) / a.n_ob));
  linear_stream_kernel<F16, NKC, G><<<dim3(unsigned(groups * a.n_ob)), dim3(kLsThreads), lds, stream>>>(a);
  RDV_HIP_TRY(hipGetLastError());
  return RDV_OK;
}

template <bool F16, int NKC>
int launch_linear_stream(const LinearStreamArgs& a, int cu, hipStream_t stream) {
  if (a.ob == kLsOutputs && a.rows * a.out >= int64_t(1) << 27) return launch_linear_stream_t<F16, NKC, 8>(a, cu, stream);
  return launch_linear_stream_t<F16, NKC, 2>(a, cu, stream);
}

__global__ __launch_bounds__(256) void relu_op_kernel(const float* __restrict__ x, float* __restrict__ y, int64_t n) {
  const int64_t n4 = n >> 2;
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  const f32x4* x4 = reinterpret_cast<const f32x4*>(x);
  f32x4* y4 = reinterpret_cast<f32x4*>(y);
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n4; i += stride) {
    f32x4 v = __builtin_nontemporal_load(x4 + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = fmaxf(v[j], 0.0f);
    __builtin_nontemporal_store(v, y4 + i);
  }
  const int64_t t = (n4 << 2) + int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0 && t < n) y[t] = fmaxf(x[t], 0.0f);
}

}  // namespace

int linear_op_check(const rdv_linear_op_desc& d, std::string* why) {
  auto bad = [&](const std::string& m) {
    *why = m;
    return RDV_ERR_INVALID;
  };
  if (d.rows < 0) return bad("rows must be >= 0");
  if (d.precision != RDV_PREC_F16 && d.precision != RDV_PREC_F32) return bad("unknown precision code");
  if (d.wkind != RDV_WKIND_F32 && d.wkind != RDV_WKIND_F16 && d.wkind != RDV_WKIND_F16_TILED16)
    return bad("unknown weight kind");
  if (d.precision == RDV_PREC_F32 && d.wkind != RDV_WKIND_F32)
    return bad("fp32 precision needs an fp32 weight");
  if (d.in_features < 8 || d.in_features % 8)
    return bad("in_features (" + std::to_string(d.in_features) + ") must be a positive multiple of 8");
  if (d.out_features < 4 || d.out_features % 4)
    return bad("out_features (" + std::to_string(d.out_features) + ") must be a positive multiple of 4");
  if (d.wkind == RDV_WKIND_F16_TILED16 && (d.in_features % 16 || d.out_features % 16))
    return bad("tiled fp16 weights need in_features and out_features multiples of 16");
  if (int64_t(d.in_features) * d.out_features >= (int64_t(1) << 31)) return bad("weight too large");
  if (d.rows >= (int64_t(1) << 40)) return bad("too many rows");
  return RDV_OK;
}

// Tile shapes of linear_gemm_kernel and the share of the matrix rate a full chip
// of them reaches (65,536 x 1024 -> 1024 fp16: 239, 310, 366, 418, 564 us; 65,536 x
// 512 -> 512 fp32: 302, 333, 347, 362, 408 us).
struct LgTile {
  int bm, bn;
  float eff16, eff32;
};
constexpr LgTile kLgTiles[] = {{256, 256, 1.0f, 1.0f}, {128, 128, 0.77f, 0.91f}, {128, 64, 0.65f, 0.87f},
                               {64, 64, 0.57f, 0.83f}, {64, 32, 0.42f, 0.74f}};

template <bool F16, bool TILED>
int launch_linear_gemm(int tile, const LinearGemmArgs& a, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_linear_gemm_t<F16, TILED, 8, 8, 4>(a, stream);
    case 1: return launch_linear_gemm_t<F16, TILED, 4, 4, 4>(a, stream);
    case 2: return launch_linear_gemm_t<F16, TILED, 4, 4, 2>(a, stream);
    case 3: return launch_linear_gemm_t<F16, TILED, 4, 2, 2>(a, stream);
    default: return launch_linear_gemm_t<F16, TILED, 4, 2, 1>(a, stream);
  }
}

int launch_linear_op(const rdv_linear_op_desc& d, const float* x, const void* w, const float* bias, float* y,
                     hipStream_t stream) {
  if (d.rows == 0) return RDV_OK;
  DeviceInfo dev;
  if (int rc = device_info(&dev)) return rc;
  const bool f16 = d.precision == RDV_PREC_F16;
  if (d.in_features <= (f16 ? 16 : 64) && d.wkind != RDV_WKIND_F16_TILED16) {
    // linear_stream_kernel where its blocks fill the chip, so many per CU that it is the
    // faster of the two (us, linear_gemm_kernel and this one, just below and at the line).
    // fp32: up to 16 columns 2 (32,768 x 8 -> 128, 1 per CU, 7.7 and 7.0; 65,536 x 8 -> 128
    // 12.3 and 9.7), to 32 4 (65,536 x 32 -> 128, 2, 12.8 and 12.9; 65,536 x 24 -> 256 21.5
    // and 19.6), to 48 2 (32,768 x 48 -> 128, 1, 10.4 and 10.5; 65,536 x 40 -> 128 17.9 and
    // 15.8), to 64 8 (32,768 x 64 -> 512, 4, 29.4 and 30.9; 65,536 x 64 -> 512 55.1 and 51.5).
    // fp16: up to 16 columns 4 (65,536 x 16 -> 128, 2, 9.8 and 9.7; 65,536 x 16 -> 256 16.9 and
    // 14.6), and past 2^18 rows, where the gemm's larger tiles write better, 32 outputs
    // (2^20 x 8 -> 32 32 and 27, 2^20 x 8 -> 64 82 and 95).  fp16 tiles, which the gemm moves by
    // DMA, are within 9% either way.
    LinearStreamArgs a = {x, w, bias, y, d.rows, 0, d.in_features, d.out_features, d.wkind, d.relu ? 1 : 0, 0, 0};
    a.tasks = (d.rows + kLsWaves * kLsRows - 1) / (kLsWaves * kLsRows);
    a.ob = std::min(kLsOutputs, (d.out_features + 15) / 16 * 16);
    a.n_ob = (d.out_features + a.ob - 1) / a.ob;
    const int chunks = (d.in_features + 15) / 16;
    const int per_cu = f16 ? 4 : chunks == 4 ? 8 : chunks == 2 ? 4 : 2;
    if (a.tasks * a.n_ob >= int64_t(per_cu) * dev.cu_count && (!f16 || d.rows <= 1 << 18 || d.out_features <= 32)) {
      if (f16) return launch_linear_stream<true, 1>(a, dev.cu_count, stream);
      if (chunks == 1) return launch_linear_stream<false, 1>(a, dev.cu_count, stream);
      if (chunks == 2) return launch_linear_stream<false, 2>(a, dev.cu_count, stream);
      if (chunks == 3) return launch_linear_stream<false, 3>(a, dev.cu_count, stream);
      return launch_linear_stream<false, 4>(a, dev.cu_count, stream);
    }
  }
  // The tile whose busiest CU has the least work: tiles per CU, rounded up, times
  // a tile's area over its efficiency.  Large products take the 256 x 256 tile,
  // small ones the one that still gives every CU a block, and none pays for a
  // last round that is nearly empty (18,624 x 512 -> 512 fp32: 122 us with 128 x
  // 128, 584 tiles; 106 us with 128 x 64).
  int best = 0;
  float cost = 0.0f;
  for (int t = 0; t < 5; ++t) {
    const LgTile& k = kLgTiles[t];
    const int64_t tiles = (d.rows + k.bm - 1) / k.bm * ((d.out_features + k.bn - 1) / k.bn);
    const float c = float((tiles + dev.cu_count - 1) / dev.cu_count) * float(k.bm * k.bn) / (f16 ? k.eff16 : k.eff32);
    if (t == 0 || c < cost) {
      best = t;
      cost = c;
    }
  }
  const LinearGemmArgs a = {x, w, bias, y, d.rows, 0, 0, d.in_features, d.out_features, 0, d.wkind, d.relu ? 1 : 0};
  if (!f16) return launch_linear_gemm<false, false>(best, a, stream);
  if (d.wkind == RDV_WKIND_F16_TILED16 && reinterpret_cast<uintptr_t>(w) % 16 == 0)
    return launch_linear_gemm<true, true>(best, a, stream);
  return launch_linear_gemm<true, false>(best, a, stream);
}

int launch_relu_op(const float* x, float* y, int64_t n, hipStream_t stream) {
  if (n == 0) return RDV_OK;
  DeviceInfo dev;
  if (int rc = device_info(&dev)) return rc;
  const int64_t n4 = std::max<int64_t>(1, n >> 2);
  const int64_t blocks = std::min<int64_t>((n4 + 255) / 256, int64_t(dev.cu_count) * 8);
  hipLaunchKernelGGL(relu_op_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, x, y, n);
  RDV_HIP_TRY(hipGetLastError());
  return RDV_OK;
}

}  // namespace rdv
