// Products of a few rows for gfx950: the linear layers and the MoE of a generation step
// (interfaces in cdx_skinny.h).
//
// With M <= 64 rows the weights are read once and used M times, so the bound is the rate
// at which the whole chip streams them.  The tile engine (cdx_gemm.h) gives one 128- or
// 256-row tile per block: a 4096-column projection of 4 rows ran on 16 of the 256 CUs.
// Here a block owns 16 NB rows of B (output columns) and its waves split K, so that a
// 4096 x 4096 operand spreads over 256 blocks of 8 waves, every wave holding up to 16 KB
// of loads in flight:
//   * B goes from global memory straight to registers as the MFMA's first operand
//     (16 rows x 32 K, 16 bytes per lane: four lanes read one 64-byte run of a row);
//     nothing is shared between waves, so LDS staging would only add a hop;
//   * A (at most 64 rows, L2-resident) is read the same way as the second operand;
//     lanes of rows past M repeat row M - 1 and their results are dropped;
//   * v_mfma_f32_16x16x32_bf16 gives C^T blocks: a lane holds one row m and four
//     consecutive columns n; the waves' partial sums meet in LDS once, at the end, and
//     are added in wave order (the same bits on every run; not those of the tile engine,
//     which adds along K in one run).
// Measured (weights from HBM, microseconds, tile engine -> here): 2048 x 2048 15.0 -> 4.1
// at 1 row, 4.7 at 8, 11.7 at 64; 4096 x 4096 27.6 -> 8.6, 9.6, 21.3 (3.9 TB/s at 1 row);
// 768 x 768 5.8 -> 2.7, 3.1, 5.7; 32000 x 2048 36.2 -> 28.9 at 1 row (4.5 TB/s), 30.4 at 8.
// MoE layers: 2048 wide, 8 experts of 704, 36.0 -> 15.2 at 4 tokens, 40.2 -> 35.9 at 64;
// 768 wide, 4 experts of 512, 18.8 -> 7.2 at 1 token, 20.4 -> 17.3 at 64.
#include "cdx_skinny.h"

namespace cdx {
namespace {

__device__ __forceinline__ bf16x8 ld8(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Operand shapes of one MFMA.  HALF (M <= 8) covers 8 output columns and 64 of K at once:
// rows 0..7 of the first operand are the columns' weights at K + 0..31 and rows 8..15 the
// same weights at K + 32..63, and the second operand likewise holds the 8 rows of A twice;
// the results are in the two diagonal quadrants and are added at the end.  Blocks are then
// half as tall (twice as many, so that 2048 columns fill 256 CUs) and A is read once per 64
// K columns instead of twice.
template <bool HALF>
struct Shape {
  static constexpr int kRows = HALF ? 8 : 16;  // output columns per MFMA
  static constexpr int kSub = HALF ? 1 : 2;    // MFMAs per 64-column chunk of K
  static __device__ __forceinline__ int row(int lane) { return HALF ? lane & 7 : lane & 15; }
  static __device__ __forceinline__ int k_off(int lane) { return (HALF ? 4 * (lane & 8) : 0) + 8 * (lane >> 4); }
};

// The waves' partial sums of one lane of one block of NI, added in wave order.
template <int NI, int W>
__device__ __forceinline__ f32x4 wave_total(const f32x4* red, int blk, int l) {
  f32x4 t = red[blk * 64 + l];
#pragma unroll
  for (int w = 1; w < W; ++w) t += red[(w * NI + blk) * 64 + l];
  return t;
}

// Result item of a block: four consecutive output columns (the q-th group of four) of one
// row m of A.  A block holds kItems of them.
template <bool HALF>
struct Item {
  static constexpr int kItems = HALF ? 16 : 64;
  int m, q;
  __device__ __forceinline__ explicit Item(int i) : m(HALF ? i & 7 : i & 15), q(HALF ? i >> 3 : i >> 4) {}
  template <int NI, int W>
  __device__ __forceinline__ f32x4 total(const f32x4* red, int blk) const {
    f32x4 t = wave_total<NI, W>(red, blk, 16 * q + m);
    if constexpr (HALF) t += wave_total<NI, W>(red, blk, 16 * (q + 2) + m + 8);
    return t;
  }
};

// RMSNorm folded into the A operand (M <= 8): the operand becomes bf16(weight * x) and the
// row's 1 / rms, a factor of the whole sum, is applied to the fp32 result, so the norm costs
// no pass of its own.  Every block reads all of x anyway and sums its squares on the way.
// (A separate norm rounds weight * x / rms to bf16 instead: the same relative rounding.)
__device__ __forceinline__ bf16x8 norm_frag(bf16x8 x, const uint4& w, float& ss) {
  float a[8], b[8];
  unpack8(__builtin_bit_cast(uint4, x), a);
  unpack8(w, b);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    ss = __builtin_fmaf(a[i], a[i], ss);
    a[i] *= b[i];
  }
  return __builtin_bit_cast(bf16x8, pack8(a));
}
// Each lane's sum of squares to the sum of its row (HALF: lanes l, l ^ 8, l ^ 16, l ^ 32 ...
// hold the row's columns), kept per wave in LDS.
__device__ __forceinline__ void row_squares(float ss, float* out, int lane) {
#pragma unroll
  for (int d = 8; d < 64; d <<= 1) ss += __shfl_xor(ss, d, 64);
  if (lane < 8) out[lane] = ss;
}
template <int W>
__device__ __forceinline__ float row_scale(const float* squares, int m, int K, float eps) {
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) t += squares[w * 8 + m];
  return rsqrtf(t / (float)K + eps);
}

// CH: 64-column chunks of K loaded before their MFMAs run (the loads in flight per wave).
// NORM: columns [0, k_split) of A enter as RMSNorm(a) (see norm_frag); their sums are kept
// apart from the second source's until the scale is applied.
template <int MT, int NB, int W, int CH, bool HALF, SkinnyEpi EPI, bool NORM = false>
__global__ __launch_bounds__(64 * W) void skinny_kernel(const SkinnyParams p) {
  using Sh = Shape<HALF>;
  constexpr int NS = Sh::kSub;
  static_assert(!NORM || (HALF && MT == 1), "the folded norm is for M <= 8");
  __shared__ f32x4 red[W * NB * MT * 64 * (NORM ? 2 : 1)];
  __shared__ float squares[NORM ? W * 8 : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = Sh::row(lane), ko = Sh::k_off(lane);
  const int n0 = blockIdx.x * (Sh::kRows * NB);

  // Element offsets of this lane's rows (the same in both K sources but for lda2).
  int64_t b_off[NB], a_off[MT], a2_off[MT];
#pragma unroll
  for (int i = 0; i < NB; ++i) b_off[i] = (int64_t)min(n0 + i * Sh::kRows + r, p.N - 1) * p.ldb + ko;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = min(i * 16 + r, p.M - 1);
    a_off[i] = (int64_t)m * p.lda + ko;
    a2_off[i] = (int64_t)m * p.lda2 + ko;
  }

  f32x4 acc[NB][MT];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 acc_n[NORM ? NB : 1];  // NORM: the sums of the normalised columns, unscaled
#pragma unroll
  for (int i = 0; i < (NORM ? NB : 1); ++i) acc_n[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss = 0.f;

  // This wave's chunks of 64 columns: one contiguous run.
  const int chunks = p.K >> 6;
  const int per = (chunks + W - 1) / W;
  const int c_end = min(chunks, (wave + 1) * per);
  for (int c0 = wave * per; c0 < c_end; c0 += CH) {
    bf16x8 bf[CH][NS][NB], af[CH][NS][MT];
    uint4 nw[NORM ? CH : 1];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (c0 + u >= c_end) break;
      const int k = (c0 + u) << 6;
      const bool second = k >= p.k_split;
      if constexpr (NORM) {
        if (!second) nw[u] = *reinterpret_cast<const uint4*>(p.norm_w + k + ko);
      }
      const uint16_t* bk = (second ? p.b2 : p.b) + (second ? k - p.k_split : k);
      const uint16_t* ak = (second ? p.a2 : p.a) + (second ? k - p.k_split : k);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
#pragma unroll
        for (int i = 0; i < NB; ++i) bf[u][s][i] = ld8(bk + b_off[i] + 32 * s);
#pragma unroll
        for (int i = 0; i < MT; ++i) af[u][s][i] = ld8(ak + (second ? a2_off[i] : a_off[i]) + 32 * s);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the batch is issued before its first use
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (c0 + u >= c_end) break;
      if constexpr (NORM) {
        if (((c0 + u) << 6) < p.k_split) {
          const bf16x8 x = norm_frag(af[u][0][0], nw[u], ss);
#pragma unroll
          for (int i = 0; i < NB; ++i) acc_n[i] = mfma16(bf[u][0][i], x, acc_n[i]);
          continue;
        }
      }
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[i][j] = mfma16(bf[u][s][i], af[u][s][j], acc[i][j]);
    }
  }

#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) red[(wave * NB * MT + i * MT + j) * 64 + lane] = acc[i][j];
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < NB; ++i) red[((W + wave) * NB + i) * 64 + lane] = acc_n[i];
    row_squares(ss, squares + wave * 8, lane);
  }
  __syncthreads();
  using It = Item<HALF>;
  for (int i = threadIdx.x; i < NB * MT * It::kItems; i += 64 * W) {
    const int blk = i / It::kItems;
    const It it(i % It::kItems);
    const int m = (blk % MT) * 16 + it.m;
    const int n = n0 + (blk / MT) * Sh::kRows + 4 * it.q;
    if (m >= p.M || n >= ((p.N + 7) & ~7)) continue;
    f32x4 t = it.template total<NB * MT, W>(red, blk);
    if constexpr (NORM)
      t += it.template total<NB, W>(red + W * NB * 64, blk) * row_scale<W>(squares, m, p.k_split, p.eps);
    float y[4] = {t[0], t[1], t[2], t[3]};
    if constexpr (EPI == SkinnyEpi::kF32) {
      *reinterpret_cast<float4*>(static_cast<float*>(p.c) + (int64_t)m * p.ldc + n) = make_float4(y[0], y[1], y[2], y[3]);
      continue;
    }
    if constexpr (EPI == SkinnyEpi::kBiasClamp) {
      const uint2 bw = *reinterpret_cast<const uint2*>(p.bias + n);
      const float bb[4] = {__uint_as_float(bw.x << 16), __uint_as_float(bw.x & 0xffff0000u),
                           __uint_as_float(bw.y << 16), __uint_as_float(bw.y & 0xffff0000u)};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v = y[j] + fminf(fmaxf(bb[j], p.bias_lo), p.bias_hi);
        y[j] = fminf(fmaxf(v, p.lo), p.hi);
      }
    }
    uint2* dst = reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.c) + (int64_t)m * p.ldc + n);
    if constexpr (EPI == SkinnyEpi::kResid || EPI == SkinnyEpi::kAccum) {
      const uint2 cw = *dst;
      const float old[4] = {__uint_as_float(cw.x << 16), __uint_as_float(cw.x & 0xffff0000u),
                            __uint_as_float(cw.y << 16), __uint_as_float(cw.y & 0xffff0000u)};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        y[j] = old[j] + (EPI == SkinnyEpi::kResid ? bf16_bits_to_f32(f32_to_bf16_bits(y[j])) : y[j]);
    }
    *dst = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
  }
}

template <int MT, int NB, int W, int CH, bool HALF>
int launch_skinny(const SkinnyParams& p, SkinnyEpi epi, hipStream_t s, const char* name) {
  constexpr int kCols = Shape<HALF>::kRows * NB;
  const dim3 grid((unsigned)((p.N + kCols - 1) / kCols)), block(64 * W);
  if constexpr (HALF) {
    if (p.norm_w != nullptr) {  // (skinny_gemm: kF32 only)
      skinny_kernel<MT, NB, W, CH, HALF, SkinnyEpi::kF32, true><<<grid, block, 0, s>>>(p);
      return check_launch(name);
    }
  }
  switch (epi) {
    case SkinnyEpi::kStore: skinny_kernel<MT, NB, W, CH, HALF, SkinnyEpi::kStore><<<grid, block, 0, s>>>(p); break;
    case SkinnyEpi::kBiasClamp:
      skinny_kernel<MT, NB, W, CH, HALF, SkinnyEpi::kBiasClamp><<<grid, block, 0, s>>>(p);
      break;
    case SkinnyEpi::kF32: skinny_kernel<MT, NB, W, CH, HALF, SkinnyEpi::kF32><<<grid, block, 0, s>>>(p); break;
    case SkinnyEpi::kResid: skinny_kernel<MT, NB, W, CH, HALF, SkinnyEpi::kResid><<<grid, block, 0, s>>>(p); break;
    default: skinny_kernel<MT, NB, W, CH, HALF, SkinnyEpi::kAccum><<<grid, block, 0, s>>>(p); break;
  }
  return check_launch(name);
}

// ---- MoE ---------------------------------------------------------------------------
// Sorted position i < T belongs to the expert whose segment [offsets[e], offsets[e + 1])
// holds it; segments are read clamped to [0, T] and permutation entries to [0, T - 1], so
// that a corrupt plan gives wrong rows but no access outside the operands.
__device__ __forceinline__ int seg_clamp(int v, int T) { return v < 0 ? 0 : (v > T ? T : v); }
__device__ __forceinline__ int row_clamp(int v, int T) { return (int)min((uint32_t)v, (uint32_t)(T - 1)); }

struct SkinnyMoeParams {
  const uint16_t* x;  // [T][H]
  const int32_t* perm;
  const int32_t* offsets;
  const uint16_t* w_gu;    // [blocks][2][P][H]
  const uint16_t* w_down;  // [blocks][H][P]
  uint16_t* inter;         // [T][S * P], rows in sorted order
  uint16_t* out;           // [T][H], rows in token order
  int32_t T, H, P, E;
  int32_t shared;          // 1: block 0 is the shared expert
  const uint16_t* norm_w;  // not null (T <= 8): the gate/up pass reads RMSNorm(x)
  float eps;
};

// Gate/up: block (unit group, weight block).  The gate and up rows of 16 (HALF: 8) units of
// one weight block times the rows of its segment, SwiGLU in the epilogue.  A routed expert
// without tokens reads nothing.
template <int MT, int W, int CH, bool HALF, bool NORM = false>
__global__ __launch_bounds__(64 * W) void skinny_gate_up_kernel(const SkinnyMoeParams p) {
  using Sh = Shape<HALF>;
  constexpr int NS = Sh::kSub;
  static_assert(!NORM || (HALF && MT == 1), "the folded norm is for T <= 8");
  __shared__ f32x4 red[W * 2 * MT * 64];
  __shared__ float squares[NORM ? W * 8 : 1];
  float ss = 0.f;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = Sh::row(lane), ko = Sh::k_off(lane);
  const bool is_shared = p.shared && blockIdx.y == 0;
  const int e = (int)blockIdx.y - p.shared;
  const int s0 = seg_clamp(p.offsets[is_shared ? 0 : e], p.T);
  const int s1 = seg_clamp(p.offsets[is_shared ? p.E : e + 1], p.T);
  const int rows = s1 - s0;
  if (rows <= 0) return;
  const int groups = (rows + 15) >> 4;  // <= MT
  const int u0 = blockIdx.x * Sh::kRows;

  const uint16_t* gate = p.w_gu + ((int64_t)blockIdx.y * 2 * p.P + u0 + r) * p.H + ko;
  const uint16_t* up = gate + (int64_t)p.P * p.H;
  // The permutation entries are on their way before the first weights and are needed after
  // them: the wait for the entries does not hold up the weights.
  int32_t src[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) src[i] = p.perm[min(s0 + i * 16 + r, s1 - 1)];

  f32x4 acc[2][MT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int chunks = p.H >> 6;
  const int per = (chunks + W - 1) / W;
  const int c_end = min(chunks, (wave + 1) * per);
  for (int c0 = wave * per; c0 < c_end; c0 += CH) {
    bf16x8 wf[CH][NS][2], xf[CH][NS][MT];
    uint4 nw[NORM ? CH : 1];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (c0 + u >= c_end) break;
      const int k = (c0 + u) << 6;
      if constexpr (NORM) nw[u] = *reinterpret_cast<const uint4*>(p.norm_w + k + ko);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        wf[u][s][0] = ld8(gate + k + 32 * s);
        wf[u][s][1] = ld8(up + k + 32 * s);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      if (j >= groups) break;
      const uint16_t* xr = p.x + (int64_t)row_clamp(src[j], p.T) * p.H + ko;
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        if (c0 + u >= c_end) break;
        const int k = (c0 + u) << 6;
#pragma unroll
        for (int s = 0; s < NS; ++s) xf[u][s][j] = ld8(xr + k + 32 * s);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (c0 + u >= c_end) break;
      if constexpr (NORM) xf[u][0][0] = norm_frag(xf[u][0][0], nw[u], ss);
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          if (j < groups) {
            acc[0][j] = mfma16(wf[u][s][0], xf[u][s][j], acc[0][j]);
            acc[1][j] = mfma16(wf[u][s][1], xf[u][s][j], acc[1][j]);
          }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) red[(wave * 2 * MT + i * MT + j) * 64 + lane] = acc[i][j];
  if constexpr (NORM) row_squares(ss, squares + wave * 8, lane);
  __syncthreads();
  const int S = 1 + p.shared;
  const int col0 = (is_shared ? 0 : p.shared * p.P) + u0;
  using It = Item<HALF>;
  for (int i = threadIdx.x; i < groups * It::kItems; i += 64 * W) {
    const int j = i / It::kItems;
    const It it(i % It::kItems);
    const int pos = s0 + j * 16 + it.m;
    if (pos >= s1) continue;
    f32x4 gv = it.template total<2 * MT, W>(red, j);
    f32x4 uv = it.template total<2 * MT, W>(red, MT + j);
    if constexpr (NORM) {
      const float rs = row_scale<W>(squares, it.m, p.H, p.eps);
      gv *= rs;
      uv *= rs;
    }
    float y[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) y[v] = silu_f32(gv[v]) * uv[v];
    *reinterpret_cast<uint2*>(p.inter + (int64_t)pos * (S * p.P) + col0 + 4 * it.q) =
        make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
  }
}

// Down: block = 16 (HALF: 8) output columns; its waves deal out the 64-column K chunks of
// every weight block in use (the shared one and the experts that have rows).  All chunks add
// into the same accumulators, a row outside a chunk's segment keeping the sum it had, so one
// bf16 rounding covers shared + routed.  (A lane's results are one row's, so the choice is
// made on them: an operand of zeros in its place would turn an Inf or NaN among one expert's
// weights into NaNs in every other expert's rows.)
template <int MT, int W, int CH, bool HALF, bool RESID>
__global__ __launch_bounds__(64 * W) void skinny_down_kernel(const SkinnyMoeParams p) {
  using Sh = Shape<HALF>;
  constexpr int NS = Sh::kSub;
  __shared__ f32x4 red[W * MT * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = Sh::row(lane), ko = Sh::k_off(lane);
  // Lane x holds expert x's segment; `left` has a bit for each expert with rows.
  const int v0 = lane < p.E ? seg_clamp(p.offsets[lane], p.T) : p.T;
  const int v1 = lane < p.E ? seg_clamp(p.offsets[lane + 1], p.T) : p.T;
  uint64_t left = __builtin_amdgcn_ballot_w64(lane < p.E && v1 > v0);
  const int first = __builtin_amdgcn_readlane(v0, 0);
  const int last = __builtin_amdgcn_readlane(v1, p.E - 1);
  if (first >= last) return;
  const int64_t ldi = (int64_t)(1 + p.shared) * p.P;
  const uint16_t* wr = p.w_down + ((int64_t)blockIdx.x * Sh::kRows + r) * p.P + ko;

  f32x4 acc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int cpb = p.P >> 6;  // chunks per weight block
  // Wave w takes chunks w, w + W, ... of the list (shared block, then the experts with
  // rows in order): c is the chunk inside the current block.
  int c = wave;
  bool sh = p.shared != 0;
  int e = -1;
  // Moves to the block that holds chunk c; false past the last one.
  auto settle = [&]() __attribute__((always_inline)) {
    if (sh) {
      if (c < cpb) return true;
      c -= cpb;
      sh = false;
    }
    while (e < 0 || c >= cpb) {
      if (e >= 0) c -= cpb;
      if (left == 0) return false;
      e = __builtin_ctzll(left);
      left &= left - 1;
    }
    return true;
  };
  bool more = settle();
  while (more) {
    bf16x8 wf[CH][NS], xf[CH][NS][MT];
    int n = 0;
    int lo[CH], hi[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      lo[u] = hi[u] = 0;
      if (more) {
        const int64_t blk = sh ? 0 : p.shared + e;
        const uint16_t* wk = wr + blk * p.H * p.P + (c << 6);
        const uint16_t* xk = p.inter + ((sh || !p.shared) ? 0 : p.P) + (c << 6) + ko;
        lo[u] = sh ? first : __builtin_amdgcn_readlane(v0, e);
        hi[u] = sh ? last : __builtin_amdgcn_readlane(v1, e);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          wf[u][s] = ld8(wk + 32 * s);
#pragma unroll
          for (int j = 0; j < MT; ++j) {
            const int pos = j * 16 + r;
            // (Rows outside the segment read a row that is written: the segment's first.)
            xf[u][s][j] = ld8(xk + (int64_t)(pos >= lo[u] && pos < hi[u] ? pos : lo[u]) * ldi + 32 * s);
          }
        }
        n = u + 1;
        c += W;
        more = settle();
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (u >= n) break;
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const int pos = j * 16 + r;
        const bool in = pos >= lo[u] && pos < hi[u];
        f32x4 t = acc[j];
#pragma unroll
        for (int s = 0; s < NS; ++s) t = mfma16(wf[u][s], xf[u][s][j], t);
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[j][v] = in ? t[v] : acc[j][v];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) red[(wave * MT + j) * 64 + lane] = acc[j];
  __syncthreads();
  using It = Item<HALF>;
  for (int i = threadIdx.x; i < MT * It::kItems; i += 64 * W) {
    const int j = i / It::kItems;
    const It it(i % It::kItems);
    const int pos = j * 16 + it.m;
    if (pos < first || pos >= last) continue;
    const f32x4 t = it.template total<MT, W>(red, j);
    const int row = row_clamp(p.perm[pos], p.T);
    uint2* dst = reinterpret_cast<uint2*>(p.out + (int64_t)row * p.H + blockIdx.x * Sh::kRows + 4 * it.q);
    uint2 o = make_uint2(pack_bf16x2(t[0], t[1]), pack_bf16x2(t[2], t[3]));
    if constexpr (RESID) {
      const uint2 c2 = *dst;
      const uint32_t a[2] = {o.x, o.y}, b[2] = {c2.x, c2.y};
      uint32_t q[2];
#pragma unroll
      for (int v = 0; v < 2; ++v)
        q[v] = pack_bf16x2(__uint_as_float(a[v] << 16) + __uint_as_float(b[v] << 16),
                           __uint_as_float(a[v] & 0xffff0000u) + __uint_as_float(b[v] & 0xffff0000u));
      o = make_uint2(q[0], q[1]);
    }
    *dst = o;
  }
}

template <int MT, int CHG, int CHD, bool HALF>
int launch_moe(const SkinnyMoeParams& p, bool residual, hipStream_t s, const char* name) {
  constexpr int W = 8, kRows = Shape<HALF>::kRows;
  const dim3 gu((unsigned)(p.P / kRows), (unsigned)(p.E + p.shared));
  if (HALF && p.norm_w != nullptr)
    skinny_gate_up_kernel<MT, W, CHG, HALF, HALF><<<gu, dim3(64 * W), 0, s>>>(p);
  else
    skinny_gate_up_kernel<MT, W, CHG, HALF><<<gu, dim3(64 * W), 0, s>>>(p);
  if (int rc = check_launch(name)) return rc;
  const dim3 grid((unsigned)(p.H / kRows));
  if (residual)
    skinny_down_kernel<MT, W, CHD, HALF, true><<<grid, dim3(64 * W), 0, s>>>(p);
  else
    skinny_down_kernel<MT, W, CHD, HALF, false><<<grid, dim3(64 * W), 0, s>>>(p);
  return check_launch(name);
}

}  // namespace

bool skinny_fits(int64_t M, int64_t N) {
  if (M > kSkinnyRows) return false;
  return M <= 16 || (M + 15) / 16 * ((N + 15) / 16) <= 4 * (int64_t)device_cu_count();
}

int skinny_gemm(const SkinnyParams& p, SkinnyEpi epi, hipStream_t s, const char* name) {
  const int cus = device_cu_count();
  if (p.norm_w != nullptr && (p.M > kNormRows || epi != SkinnyEpi::kF32))
    return fail(CDX_EUNSUPPORTED, "%s: a folded norm needs M <= 8", name);
  // The columns per block grow with N: one MFMA's worth while that fills the chip at most
  // once, more for wider outputs (fewer blocks and A reads for the same loads in flight).
  // us on 256 CUs, weights from HBM.  8 rows, K = 2048, blocks of 8 / 16 / 32 columns: N = 2048 4.7 /
  // 5.5 / 7.2, 4096 6.5 / 6.0 / 7.5, 8192 10.3 / 9.1 / 10.0, 32000 35.0 / 30.0 / 30.7 (K = 768: 16.2 /
  // 13.3 / 12.0).  16 rows, blocks of 16 / 64: N = 4096 6.5 / 11.9, 8192 10.4 / 12.7, 12288 14.9 / 14.0,
  // 32000 35.9 / 33.2.
  if (p.M <= 8) {
    if (p.N <= 8 * cus) return launch_skinny<1, 1, 8, 8, true>(p, epi, s, name);
    if (p.N <= 32 * cus) return launch_skinny<1, 2, 8, 4, true>(p, epi, s, name);
    return launch_skinny<1, 4, 8, 4, true>(p, epi, s, name);
  }
  if (p.M <= 16) {
    if (p.N <= 32 * cus) return launch_skinny<1, 1, 8, 4, false>(p, epi, s, name);
    return launch_skinny<1, 4, 8, 2, false>(p, epi, s, name);
  }
  if (p.M <= 32) return launch_skinny<2, 1, 8, 4, false>(p, epi, s, name);
  return launch_skinny<4, 1, 8, 2, false>(p, epi, s, name);
}

int skinny_moe(const uint16_t* x, int32_t T, int32_t H, int32_t P, int32_t E, bool shared, const int32_t* perm,
               const int32_t* offsets, const uint16_t* w_gu, const uint16_t* w_down, uint16_t* inter, uint16_t* out,
               bool residual, const uint16_t* norm_w, float eps, hipStream_t s, const char* name) {
  SkinnyMoeParams p{x, perm, offsets, w_gu, w_down, inter, out, T, H, P, E, shared ? 1 : 0, norm_w, eps};
  if (norm_w != nullptr && T > kNormRows) return fail(CDX_EUNSUPPORTED, "%s: a folded norm needs T <= 8", name);
  if (T <= 8) return launch_moe<1, 4, 4, true>(p, residual, s, name);
  if (T <= 16) return launch_moe<1, 4, 4, false>(p, residual, s, name);
  if (T <= 32) return launch_moe<2, 2, 4, false>(p, residual, s, name);
  return launch_moe<4, 2, 2, false>(p, residual, s, name);
}

}  // namespace cdx
