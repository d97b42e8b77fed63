// The training step of a narrow chain in one kernel: forward, loss and backward
// of each 32-point tile in registers, no activation or gradient through memory.
//
// For chains whose hidden layers are all 32 or all 64 wide, with at most 64
// inputs and 16 outputs, a wave can hold everything a tile needs: D hidden
// activations as the matrix-core fragments the next layer reads (16 registers
// each at 64), and the fp32 dW of every layer (16 registers per 32 x 32 block; 256
// for 32 -> 64 x 4 -> 16, so one wave per SIMD).  Per tile:
//   forward: H^T = W X^T per layer (mlp_layout.h's fragments and hand-off, the
//     sequence of train_fwd_kernel, so h is the same to the bit);
//   head: g = 2 (y - t), the loss;
//   backward, layer by layer from the head: g^T and h^T as K = points operands
//     (through the wave's LDS scratch: point-major in, transposing reads out), dW +=
//     g^T h and db in registers, g_{l-1}^T = W^T g^T masked by h > 0 (W^T fragments
//     in LDS).
// At the end a block sums its waves' dW through LDS and writes one partial.
//
// Bound: the vector ALU's hand-offs, masks and conversions plus the matrix cores
// (90 MFMAs, 2,880 cycles, per tile of 32 -> 64 x 4 -> 16), which add up at one wave
// per SIMD.  262,144 points of that chain, whole step: 209 us with a kernel per
// layer pair (run-time shapes, transposes by 2-byte LDS writes, activations through
// memory) -> 51 us (dW in accumulation registers, packed masks, weights fetched a
// stage ahead, one reduction launch, one round trip of staging).  Transposing by
// products with 0/1 fragments takes 35 more MFMAs, the same time (51.0 us, here
// 50.5; 1 to 2 layers 4 to 10% less at 2^19 points, 5 layers of 32 8% more) and
// turns one infinity or NaN into NaN across its 32 features.
#include <algorithm>

#include "train_fused.h"
#include "train_tile.h"

namespace rdv {

struct TrainFusedArgs {
  const uint8_t* packed;
  const half_t* x;        // [n, in]
  const float* target;    // [n, out]
  float* loss_partial;    // [gridDim.x]
  float* dw[kTrainFusedDepth + 1];  // [gridDim.x][out][in] per layer
  float* db[kTrainFusedDepth + 1];  // [gridDim.x][out]
  int64_t frag_off[kTrainFusedDepth + 1], bias_off[kTrainFusedDepth + 1], w32_off[kTrainFusedDepth + 1];
  int64_t n;
  int in, out, kc0;
};

constexpr int fused_waves(int mt) { return mt == 1 ? 8 : 4; }  // per block

// Shapes: D hidden layers of 32 MT, 2 MTI K chunks of input (a missing chunk is
// zeros), a head of at most 16 outputs.
template <int MT, int D, int MTI>
struct FusedNet {
  static constexpr int kNW = fused_waves(MT);
  static constexpr int kKC = 2 * MT;              // K chunks of a hidden width
  static constexpr int kKC0 = 2 * MTI;
  // forward fragments (1 KiB units): layer 0 [MT][KC0], hidden [MT][KC] each, head [1][KC]
  static constexpr int fw(int l) { return l == 0 ? 0 : MT * kKC0 + (l - 1) * MT * kKC; }
  static constexpr int kFw = fw(D) + kKC;
  // transposed fragments: layers 1 .. D - 1 [MT][KC], head [MT][1]
  static constexpr int wt(int l) { return kFw + (l - 1) * MT * kKC; }
  static constexpr int kUnits = wt(D) + MT;
  static constexpr int kBias = 32 * (D * MT + 1);
  // dW accumulators (32 x 32 blocks): layer 0 [MT][MTI], hidden [MT][MT] each, head [1][MT]
  static constexpr int dw(int l) { return l == 0 ? 0 : MT * MTI + (l - 1) * MT * MT; }
  static constexpr int kAcc = dw(D) + MT;
  // Blocks held in accumulation registers, of which a wave has 256 (fused_dw): the
  // first 16.  Any after those (the head's, at 64 wide, 4 deep and past 32 inputs) are
  // ordinary registers.
  static constexpr int kAgpr = kAcc < 16 ? kAcc : 16;
  static_assert(kAgpr * 16 <= 256 && kAcc - kAgpr <= 2, "dW in registers");
  // stages of a tile, each with its weight fragments: forward layers 0 .. D (the
  // head), then the transposed ones of layers D .. 1
  static constexpr int kStages = 2 * D + 1;
  static constexpr int st_base(int s) { return s <= D ? fw(s) : wt(2 * D + 1 - s); }
  static constexpr int st_units(int s) { return s < D ? (s == 0 ? MT * kKC0 : MT * kKC) : s == D ? kKC : s == D + 1 ? MT : MT * kKC; }
  static constexpr int kStMax = MT * (kKC > kKC0 ? kKC : kKC0);
  // a wave's transposing scratch: g_l and h_{l-1} of its tile, a row of 128 bytes per point
  static constexpr int kTr = 32 * 128;
  static constexpr int kTrOff = kUnits * 1024 + kBias * 4;
  static constexpr int kLds = kTrOff + kNW * 3 * kTr;
  static constexpr int kRB = 4;                   // accumulator blocks summed per round at the end
  static constexpr int kRed = kRB * kNW * 4096;
  static constexpr int kBytes = kLds > kRed ? kLds : kRed;
  static_assert(kBytes <= 150 * 1024, "LDS");
};

// g where h > 0, else +0, two halves per instruction (the compiler turns the same
// expression into a compare and a select per half): h's bits as signed integers
// clamped to 0 .. 1, negated to a mask.
__device__ __forceinline__ half8 fused_mask(const half8& g, const half8& h) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 hb = __builtin_bit_cast(u32x4, h), gb = __builtin_bit_cast(u32x4, g);
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t m, hi = hb[i];
    asm("v_pk_max_i16 %0, %1, 0\n\t"
        "v_pk_min_i16 %0, %0, %2\n\t"
        "v_pk_sub_i16 %0, 0, %0"
        : "=&v"(m)
        : "v"(hi), "s"(0x00010001u));
    r[i] = gb[i] & m;
  }
  return __builtin_bit_cast(half8, r);
}

// acc += a0 b0 + a1 b1 with acc in accumulation registers.  Written out so that
// only the dW blocks live there: the compiler's own choice, made for a whole
// function, puts the short-lived products there too and then moves every value
// back before its conversion (560 moves per tile).  The compiler does not know
// these for products and puts no wait before an access of acc: nothing else may
// touch it inside the tile loop, so the blocks must fit the file (kAgpr; a 17th
// makes the compiler move blocks in and out between products), and
// fused_dw_done ends every tile.
__device__ __forceinline__ void fused_dw(f32x16& acc, const half8& a0, const half8& b0, const half8& a1, const half8& b1) {
  asm volatile(
      "s_nop 1\n\t"
      "v_mfma_f32_32x32x16_f16 %0, %1, %2, %0\n\t"
      "v_mfma_f32_32x32x16_f16 %0, %3, %4, %0"
      : "+a"(acc)
      : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
}
// The wait a read of acc needs after its last product, at the end of each tile
// (32 of its ~10,000 cycles); every later read depends on it.
template <int N>
__device__ __forceinline__ void fused_dw_done(f32x16 (&acc)[N]) {
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+a"(acc[i]));
}

// A wave's transposing scratch: a row of 128 bytes per point, 32-byte slots (slot s:
// features 16 s ..).  A row's slots are permuted by its last two bits and their
// 16-byte halves by the third, so that the 8 lanes of a 16-byte write and the 16 of
// a transposing read (4 rows x 32 bytes) each find different banks; slot s is at
// the offset of slot 0 xor 32 s.
__device__ __forceinline__ uint32_t fused_slot(int point, int s, int half) {
  return uint32_t(point * 128 + ((s ^ (point & 3)) << 5) + ((half ^ ((point >> 2) & 1)) << 4));
}

// 8 points of a feature per lane as half a K = points operand: elements j: points
// tfl_feature(0, hh, j) past the first row.  src: the lane's piece of its quartet of
// rows; a transposing read hands lane i of 16 column i of the block of 4 x 16 values
// whose 8-byte pieces the lanes point at, lane i at piece i % 4 of row i / 4.
__device__ __forceinline__ half8 fused_points(uint32_t src) {
  typedef __fp16 tf_half4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) tf_half4 lds_h4;
  const half4v lo = __builtin_bit_cast(half4v, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4*)(src)));
  const half4v hi = __builtin_bit_cast(half4v, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4*)(src + 8 * 128)));
  return half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

template <int MT, int D, int MTI>
__global__ __launch_bounds__(64 * fused_waves(MT), 1) void train_fused_kernel(TrainFusedArgs a) {
  using N = FusedNet<MT, D, MTI>;
  constexpr int KC = N::kKC, KC0 = N::kKC0, NW = N::kNW, T = 64 * NW, H = 32 * MT;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ float s_loss[NW];
  __shared__ float s_db[NW][32 * (D * MT + 1)];
  half8* const sw = reinterpret_cast<half8*>(smem);
  float* const sb = reinterpret_cast<float*>(smem + N::kUnits * 1024);
  const int tid = int(threadIdx.x), lane = tid & 63, h = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t n = a.n, ntiles = (n + 31) / 32;
  const int in = a.in, out = a.out;

  const int64_t per = (ntiles + gridDim.x - 1) / gridDim.x;
  const int64_t t_begin = int64_t(blockIdx.x) * per;
  const int64_t t_end = t_begin + per < ntiles ? t_begin + per : ntiles;
  half8 bx[KC0], nx[KC0];
  auto load_x = [&](int64_t tile, half8 (&b)[KC0]) {
    const int64_t p = tile * 32 + col;
    const half_t* row = a.x + (p < n ? p : n - 1) * in + 8 * h;
#pragma unroll
    for (int c = 0; c < KC0; ++c) b[c] = *reinterpret_cast<const half8*>(row + 16 * (c < a.kc0 ? c : 0));
  };
  if (t_begin + wave < t_end) load_x(t_begin + wave, nx);

  // ---- parameters: forward fragments, transposed fragments from the fp32 copy,
  // biases.  Every load goes out before the first LDS write (a block starts once
  // per call, and a load waited for in a loop costs a memory latency per turn).
  {
    constexpr int FI = (N::kFw * 64 + T - 1) / T, WI = (MT * KC * 64 + T - 1) / T, BI = (N::kBias + T - 1) / T;
    half8 fr[FI];
#pragma unroll
    for (int k = 0; k < FI; ++k) {
      const int i = min(k * T + tid, N::kFw * 64 - 1), u = i >> 6;
      if (u < MT * KC0) {
        const int t = u / KC0, c = u % KC0;
        fr[k] = reinterpret_cast<const half8*>(a.packed + a.frag_off[0])[(t * a.kc0 + (c < a.kc0 ? c : 0)) * 64 + (i & 63)];
        if (c >= a.kc0) fr[k] = half8{};
      } else {
        const int l = min(1 + (u - MT * KC0) / (MT * KC), D);
        fr[k] = reinterpret_cast<const half8*>(a.packed + a.frag_off[l])[i - N::fw(l) * 64];
      }
    }
    float wv[D][WI][8];
#pragma unroll
    for (int l = 1; l <= D; ++l) {
      const float* w32 = reinterpret_cast<const float*>(a.packed + a.w32_off[l]);
      const int kc = l == D ? 1 : KC, ow = l == D ? out : H;
#pragma unroll
      for (int k = 0; k < WI; ++k) {
        if (k * T < MT * kc * 64) {
          const int i = min(k * T + tid, MT * kc * 64 - 1);
          const int t = (i >> 6) / kc, c = (i >> 6) % kc;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int o = tfl_feature(c, (i >> 5) & 1, e);
            const float w = w32[(o < ow ? o : 0) * H + 32 * t + (i & 31)];
            wv[l - 1][k][e] = o < ow ? w : 0.0f;
          }
        }
      }
    }
    float bv[BI];
#pragma unroll
    for (int k = 0; k < BI; ++k) {
      const int i = min(k * T + tid, N::kBias - 1), l = min(i / H, D);
      bv[k] = reinterpret_cast<const float*>(a.packed + a.bias_off[l])[i - l * H];
    }
    // spare threads rewrite the last element (same value)
#pragma unroll
    for (int k = 0; k < FI; ++k) sw[min(k * T + tid, N::kFw * 64 - 1)] = fr[k];
#pragma unroll
    for (int l = 1; l <= D; ++l) {
      const int kc = l == D ? 1 : KC;
#pragma unroll
      for (int k = 0; k < WI; ++k) {
        if (k * T < MT * kc * 64) {
          half8 v;
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = half_t(wv[l - 1][k][e]);
          sw[N::wt(l) * 64 + min(k * T + tid, MT * kc * 64 - 1)] = v;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < BI; ++k) sb[min(k * T + tid, N::kBias - 1)] = bv[k];
  }
  // the wave's scratch (g's part, then two of h's): this lane's point, and its piece of a transposing read
  typedef __attribute__((address_space(3))) half8 lds_h8;
  const uint32_t tg = uint32_t(reinterpret_cast<uintptr_t>(smem + N::kTrOff + wave * 3 * N::kTr));
  const uint32_t put0 = fused_slot(col, 0, h);
  const uint32_t get0 = fused_slot(4 * h + ((lane >> 2) & 3), (lane >> 4) & 1, (lane >> 1) & 1) + 8 * (lane & 1);
  __syncthreads();

  f32x16 acc[N::kAgpr], accv[N::kAcc > N::kAgpr ? N::kAcc - N::kAgpr : 1];
#pragma unroll
  for (int i = 0; i < N::kAgpr; ++i) acc[i] = f32x16{};
#pragma unroll
  for (int i = N::kAgpr; i < N::kAcc; ++i) accv[i - N::kAgpr] = f32x16{};
  float db[D * MT + 1];
#pragma unroll
  for (int i = 0; i <= D * MT; ++i) db[i] = 0.0f;
  float loss = 0.0f;

  for (int64_t tile = t_begin + wave; tile < t_end; tile += NW) {
    const half8* ws = sw + opaque_zero() + lane;
    const float* bs = sb + opaque_zero();
    const int64_t p = tile * 32 + col;
    const bool pv = p < n;
    f32x4 tv[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int r = 8 * q < out ? 8 * q : 0;
      tv[q] = *reinterpret_cast<const f32x4*>(a.target + (pv ? p : n - 1) * out + r + 4 * h);
    }
#pragma unroll
    for (int c = 0; c < KC0; ++c) bx[c] = c < a.kc0 && pv ? nx[c] : half8{};  // points past n: no input, no gradient
    if (tile + NW < t_end) load_x(tile + NW, nx);

    // The next stage's fragments are read while this one computes (the wave is
    // alone on its SIMD: a read waited for at its use costs its whole latency).
    half8 wb[2][N::kStMax];
    auto fetch = [&](int st) {
#pragma unroll
      for (int u = 0; u < N::kStMax; ++u)
        if (st < N::kStages && u < N::st_units(st)) wb[st & 1][u] = ws[(N::st_base(st) + u) * 64];
      __builtin_amdgcn_sched_barrier(0);
    };
    fetch(0);

    half8 b[D][KC];
    // g's slot s, and layer l's input h_{l-1} (two buffers), point-major into the
    // scratch; the wave's own LDS accesses stay in order
    auto put_g = [&](int s, const half8& v) { *(lds_h8*)(tg + ((put0 + opaque_zero()) ^ (32 * s))) = v; };
    auto put_h = [&](int l) {
      const uint32_t put = put0 + opaque_zero();
#pragma unroll
      for (int s = 0; s < (KC > KC0 ? KC : KC0); ++s)
        if (s < (l == 0 ? KC0 : KC))
          *(lds_h8*)(tg + (put ^ (32 * s)) + (1 + (l & 1)) * N::kTr) = l == 0 ? bx[s < KC0 ? s : 0] : b[l > 0 ? l - 1 : 0][s < KC ? s : 0];
    };

    // ---- forward
    auto bias = [&](int base) {
      f32x16 v;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(bs + base + 8 * q + 4 * h);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[4 * q + j] = x[j];
      }
      return v;
    };
#pragma unroll
    for (int l = 0; l < D; ++l) {
      fetch(l + 1);
      f32x16 y[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) y[t] = bias(l * H + 32 * t);
      const int kc = l == 0 ? KC0 : KC;
#pragma unroll
      for (int c = 0; c < (l == 0 ? KC0 : KC); ++c)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          y[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb[l & 1][t * kc + c], l == 0 ? bx[c < KC0 ? c : 0] : b[l > 0 ? l - 1 : 0][c < KC ? c : 0], y[t], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < KC; ++s) {
        half8 v = tp2_half(y[s / 2], s & 1);
        b[l][s] = __builtin_elementwise_max(v, half8{0, 0, 0, 0, 0, 0, 0, 0});
      }
    }
    // ---- head: rows 8 hi + 4 h + jj < out of D; g = 2 (y - t) as one slot
    half8 g[KC];
    {
      fetch(D + 1);
      put_h(D);
      f32x16 y = bias(D * H);
#pragma unroll
      for (int c = 0; c < KC; ++c)
        y = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb[D & 1][c], b[D - 1][c], y, 0, 0, 0);
#pragma unroll
      for (int hi = 0; hi < 2; ++hi) {
        const bool ok = 8 * hi < out && pv;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float d = ok ? y[4 * hi + j] - tv[hi][j] : 0.0f;
          loss += d * d;
          g[0][4 * hi + j] = half_t(d + d);
        }
      }
      put_g(0, g[0]);
    }
    // ---- backward
#pragma unroll
    for (int l = D; l >= 0; --l) {
      fetch(2 * D + 2 - l);
      // back as K = points operands.  Moved, not multiplied by a 0/1 selection: an
      // infinity or a NaN of one feature must not reach the others.
      const uint32_t get = get0 + opaque_zero();
      half8 ht[MT > MTI ? MT : MTI][2], gt[MT][2];
#pragma unroll
      for (int t = 0; t < (l == 0 ? MTI : MT); ++t)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) ht[t][ks] = fused_points(tg + (get ^ (64 * t)) + (1 + (l & 1)) * N::kTr + 16 * ks * 128);
#pragma unroll
      for (int o = 0; o < (l == D ? 1 : MT); ++o)  // (the head's rows past 16 are whatever slot 1 holds: never stored)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) gt[o][ks] = fused_points(tg + (get ^ (64 * o)) + 16 * ks * 128);
      f32x16 d[MT];
      if (l > 0) {
        put_h(l - 1);
#pragma unroll
        for (int t = 0; t < MT; ++t) d[t] = f32x16{};
#pragma unroll
        for (int c = 0; c < (l == D ? 1 : KC); ++c)
#pragma unroll
          for (int t = 0; t < MT; ++t)
            d[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb[(2 * D + 1 - l) & 1][t * (l == D ? 1 : KC) + c], g[c], d[t], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      // dW_l and db, and between their products g_{l-1}
      auto mask = [&](int s) {
        g[s] = fused_mask(tp2_half(d[s / 2], s & 1), b[l > 0 ? l - 1 : 0][s]);
        put_g(s, g[s]);
      };
      constexpr int kPairs = MT * (MT > MTI ? MT : MTI);
#pragma unroll
      for (int i = 0; i < kPairs; ++i) {
        const int mi = l == 0 ? MTI : MT, o = i / mi, t = i % mi;
        if (o < (l == D ? 1 : MT)) {
          if (t == 0) db[l * MT + o] = tp2_sum(gt[o][1], tp2_sum(gt[o][0], db[l * MT + o]));
          const int k = N::dw(l) + o * mi + t;
          if (k < N::kAgpr) {
            fused_dw(acc[k < N::kAgpr ? k : 0], gt[o][0], ht[t][0], gt[o][1], ht[t][1]);
          } else {
            f32x16& v = accv[k < N::kAgpr ? 0 : k - N::kAgpr];
            v = __builtin_amdgcn_mfma_f32_32x32x16_f16(gt[o][0], ht[t][0], v, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_32x32x16_f16(gt[o][1], ht[t][1], v, 0, 0, 0);
          }
        }
        if (l > 0 && i < KC) mask(i);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (l > 0) {
#pragma unroll
        for (int s = kPairs; s < KC; ++s) mask(s);
      }
    }
    fused_dw_done(acc);
  }

  // ---- the block's sums: loss, db, then dW in rounds of RB blocks (every wave
  // writes its RB blocks to LDS, wave w sums block w over the waves in order)
  constexpr int RB = N::kRB;
  loss = tr_wave_sum(loss);
  if (lane == 0) s_loss[wave] = loss;
#pragma unroll
  for (int i = 0; i <= D * MT; ++i) {
    const float v = db[i] + __shfl_xor(db[i], 32, 64);
    if (h == 0) s_db[wave][32 * i + hidden_slot_feature(col)] = v;  // lane col summed position col of its block
  }
  f32x4* const red = reinterpret_cast<f32x4*>(smem);  // [block][wave][4][64]
#pragma unroll
  for (int k0 = 0; k0 < N::kAcc; k0 += RB) {
    __syncthreads();  // the weights, or the previous round, are no longer read
#pragma unroll
    for (int k = 0; k < RB; ++k) {
      if (k0 + k < N::kAcc) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int b = k0 + k;
          const f32x16& v = b < N::kAgpr ? acc[b < N::kAgpr ? b : 0] : accv[b < N::kAcc && b >= N::kAgpr ? b - N::kAgpr : 0];
          red[((k * NW + wave) * 4 + q) * 64 + lane] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
        }
      }
    }
    __syncthreads();
    const int k = k0 + wave;
    if (wave < RB && k < N::kAcc) {
      int l = 0;
#pragma unroll
      for (int i = 1; i <= D; ++i) l = k >= N::dw(i) ? i : l;
      const int r = k - (l == 0 ? 0 : MT * MTI + (l - 1) * MT * MT);
      const int mi = l == 0 ? MTI : MT, iw = l == 0 ? in : H, ow = l == D ? out : H;
      float* dst = a.dw[l] + int64_t(blockIdx.x) * ow * iw;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 s = red[(wave * NW * 4 + q) * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) s += red[((wave * NW + w) * 4 + q) * 64 + lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // positions to features: g and h in the hidden order, x in its own
          const int o = hidden_slot_feature(32 * (r / mi) + 8 * q + 4 * h + j);
          const int i = l == 0 ? 32 * (r % mi) + col : hidden_slot_feature(32 * (r % mi) + col);
          if (o < ow && i < iw) dst[int64_t(o) * iw + i] = s[j];
        }
      }
    }
  }
  if (tid == 0) {
    float s = 0.0f;
    for (int w = 0; w < NW; ++w) s += s_loss[w];
    a.loss_partial[blockIdx.x] = s;
  }
  for (int i = tid; i < N::kBias; i += T) {
    float s = 0.0f;
    for (int w = 0; w < NW; ++w) s += s_db[w][i];
    const int l = min(i / H, D), o = i - l * H, ow = l == D ? out : H;
    if (o < ow) a.db[l][int64_t(blockIdx.x) * ow + o] = s;
  }
}

struct FusedKernel {
  const void* fn;
  int waves, bytes;
};

template <int MT, int D, int MTI>
FusedKernel fused_entry() {
  using N = FusedNet<MT, D, MTI>;
  return {reinterpret_cast<const void*>(&train_fused_kernel<MT, D, MTI>), N::kNW, N::kBytes};
}

static const FusedKernel* fused_kernel(int mt, int depth, int mti) {
  static const FusedKernel k1[5][2] = {{fused_entry<1, 1, 1>(), fused_entry<1, 1, 2>()},
                                       {fused_entry<1, 2, 1>(), fused_entry<1, 2, 2>()},
                                       {fused_entry<1, 3, 1>(), fused_entry<1, 3, 2>()},
                                       {fused_entry<1, 4, 1>(), fused_entry<1, 4, 2>()},
                                       {fused_entry<1, 5, 1>(), fused_entry<1, 5, 2>()}};
  static const FusedKernel k2[4][2] = {{fused_entry<2, 1, 1>(), fused_entry<2, 1, 2>()},
                                       {fused_entry<2, 2, 1>(), fused_entry<2, 2, 2>()},
                                       {fused_entry<2, 3, 1>(), fused_entry<2, 3, 2>()},
                                       {fused_entry<2, 4, 1>(), fused_entry<2, 4, 2>()}};
  if (mt == 1 && depth <= 5) return &k1[depth - 1][mti - 1];
  if (mt == 2 && depth <= 4) return &k2[depth - 1][mti - 1];
  return nullptr;
}

// The chain's kernel, or nullptr: equal hidden widths of 32 (up to 5 layers) or
// 64 (up to 4: a fifth's dW fits no registers, FusedNet::kAgpr), at most 64 inputs and
// 16 outputs.
static const FusedKernel* fused_for(const rdv_mlp_desc& d) {
  const int L = d.n_layers, hw = d.dims[1];
  if (L < 2 || L > kTrainFusedDepth + 1 || (hw != 32 && hw != 64) || d.dims[0] > 64 || d.dims[L] > 16) return nullptr;
  for (int l = 1; l < L; ++l)
    if (d.dims[l] != hw) return nullptr;
  return fused_kernel(hw / 32, L - 1, (d.dims[0] + 31) / 32);
}

bool train_fused_ok(const rdv_mlp_desc& d) { return fused_for(d) != nullptr; }

int train_fused_blocks(const rdv_mlp_desc& d, int64_t n, int cu) {
  const FusedKernel* k = fused_for(d);
  return int(std::max<int64_t>(1, std::min<int64_t>(cu, ((n + 31) / 32 + k->waves - 1) / k->waves)));
}

int launch_train_fused(const rdv_mlp_desc& d, const MlpLayout& lay, const void* packed, const void* x,
                       const float* target, int64_t n, int blocks, float* loss_partial, float* const* dw,
                       float* const* db, hipStream_t stream) {
  const FusedKernel* k = fused_for(d);
  TrainFusedArgs a = {};
  a.packed = static_cast<const uint8_t*>(packed);
  a.x = static_cast<const half_t*>(x);
  a.target = target;
  a.loss_partial = loss_partial;
  for (int l = 0; l < d.n_layers; ++l) {
    a.dw[l] = dw[l];
    a.db[l] = db[l];
    a.frag_off[l] = lay.frag_off[l];
    a.bias_off[l] = lay.bias_off[l];
    a.w32_off[l] = lay.w32_off[l];
  }
  a.n = n;
  a.in = d.dims[0];
  a.out = d.dims[d.n_layers];
  a.kc0 = lay.kc[0];
  RDV_HIP_TRY(hipFuncSetAttribute(k->fn, hipFuncAttributeMaxDynamicSharedMemorySize, k->bytes));
  void* args[] = {&a};
  RDV_HIP_TRY(hipLaunchKernel(k->fn, dim3(unsigned(blocks)), dim3(unsigned(64 * k->waves)), args, size_t(k->bytes), stream));
  return RDV_OK;
}

}  // namespace rdv
