// Pair transition (Protenix Transition, n = 4, c = 128) on the CDNA4 16-bit
// matrix cores, FP32-accurate:
//
//   h   = silu(LN(x) W_a^T) * (LN(x) W_b^T)       [rows][512]
//   out = h W_o^T  (or out + h W_o^T, the residual)  [rows][128]
//
// One fused kernel with h never leaving the registers
// (transition_fused_kernel below), after a small kernel that folds the
// LayerNorm affine into the weights and splits them into scaled fp16 planes.
#include "attn_common.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "split.hpp"

#include <algorithm>
#include <type_traits>

namespace fpx {
namespace {

constexpr int kHid = kTransitionHidden;

// ------------------------------------------------------- fused, fp16 cores
// out = x + silu(y Wa'^T + ba) * (y Wb'^T + bb) Wo^T with y = (x - mean)
// rstd, the LayerNorm affine folded into the weights (W' = W diag(ln_w),
// b = W ln_b), all three products on v_mfma_f32_32x32x16_f16 with
// power-of-two scaled fp16 (hi, lo) planes and three terms (FP32 accuracy).
// A wave owns 32 pair rows: its y^T planes (the B operand, 64 VGPRs) stay in
// registers while the 512 hidden channels pass in 16 chunks of 32; per chunk
//   value^T, gate^T [32 hidden][32 rows] = W' y^T      (48 MFMAs)
//   h = silu(gate) * value, as planes scaled by 2^e_h  (the A operand: a
//       lane holds its row's 16 hidden values, and W_o's columns are stored
//       in that order)
//   out [32 rows][128] += h W_o^T                       (24 MFMAs)
// so h never leaves the registers.  The chunks' weight planes (48 KB each,
// written once per call by transition_prep_kernel) go from L2 into an LDS
// ring by global_load_lds, shared by the 8 waves (256 rows) of a work-group,
// with one barrier per chunk.  Plane scales: y by 2^e_x
// (|y_c| <= sqrt(128)), each row of W' and of W_o by its own exponent, h by
// 2^e_h from the bound |h_c| <= max(|g_c|, 0.2785) |v_c| with |g_c| <=
// sqrt(128) |Wa'_c| + |ba_c| (likewise v), |silu(g)| <= max(|g|, 0.2785).
constexpr int kFusedWaves = 8;
constexpr int kFusedRows = 32 * kFusedWaves;               // rows per tile
constexpr int kChunkHid = 32;
constexpr int kChunks = kHid / kChunkHid;                  // 16
constexpr int kUpBlocks = 2 * 8 * 2;                       // [a, b][k step][hi, lo]
constexpr int kDownBlocks = 4 * 2 * 2;                     // [out block][k step][hi, lo]
constexpr int kPlaneBlock = 32 * 16;                       // fp16 values of a 1 KB block
constexpr int kChunkValues = (kUpBlocks + kDownBlocks) * kPlaneBlock;  // 24576 (48 KB)
constexpr int kChunkBytes = kChunkValues * 2;

// Plane exponents (TransitionArgs::exps): e_x of the y planes, one per W' row
// (a, then b) and one per W_o row; then the prep work-groups' largest h
// bounds (float bits), which the fused kernel reduces to e_h.
constexpr int kExpX = 0;
constexpr int kExpW = 4;                 // [2][512]
constexpr int kExpO = kExpW + 2 * kHid;  // [128]
constexpr int kPrepUp = kHid / 16;           // work-groups of 16 hidden channels
constexpr int kPrepDown = kChannels / 8;     // work-groups of 8 W_o rows
constexpr int kExpPart = kExpO + kChannels;  // [kPrepUp]

// The folded biases ([2][512]: ba, bb), the exponents and the weight planes.
// Work-group g < kPrepUp: hidden channels 16 g .. + 15 (a and b rows, eight
// threads per row, 16 inputs each); the others: W_o rows 8 g' .. + 7 (32
// threads per row, 16 values each).  Every work-group holds whole rows, so
// their exponents need no other work-group: one launch of one load phase
// (5.4 us) where exponents and planes were two (9.3 + 5.1 us).
//
// Planes of chunk c:
//   up   [a, b][k step t][hi, lo][k / 8][hidden m][k % 8]: W'[32 c + m][16 t + k] 2^e_w
//   down [out block ob][k step s][hi, lo][k / 8][out o][k % 8]: W_o[32 ob + o][32 c +
//        16 s + 8 (k / 4 % 2) + 4 (k / 8) + k % 4] 2^e_o, the hidden order in
//        which a lane of the value^T / gate^T results holds its row's values.
// A 1 KB block's two halves are the k / 8 halves, so the 32 lanes of a half
// read 512 contiguous bytes (no LDS bank conflicts).
__global__ __launch_bounds__(256) void transition_prep_kernel(TransitionArgs a) {
  const int tid = threadIdx.x;
  if ((int)blockIdx.x >= kPrepUp) {
    const int o = ((int)blockIdx.x - kPrepUp) * 8 + (tid >> 5);
    const int part = tid & 31;  // hidden channels 16 part .. + 15: k step part % 2 of chunk part / 2
    const float* src = a.w_o + (int64_t)o * kHid + 16 * part;
    f32x4 v[4];
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = *(const f32x4*)(src + 4 * i);
      m = __builtin_elementwise_maximum(
          m, __builtin_elementwise_maximum(
                 __builtin_elementwise_maximum(__builtin_fabsf(v[i].x), __builtin_fabsf(v[i].y)),
                 __builtin_elementwise_maximum(__builtin_fabsf(v[i].z), __builtin_fabsf(v[i].w))));
    }
    const int e = plane_exp(half_max(m));
    if (part == 0) a.exps[kExpO + o] = e;
    __bf16* dst = a.planes + (int64_t)(part >> 1) * kChunkValues + kUpBlocks * kPlaneBlock +
                  (((o >> 5) * 2 + (part & 1)) * 2) * kPlaneBlock + (o & 31) * 8;
    // k half kh holds values 4 kh .. + 3 and 8 + 4 kh .. + 3
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      const f32x4 p = v[kh], q = v[2 + kh];
      bf16x8 hi, lo;
      split_f16(ldexp8(f32x8{p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w}, e), hi, lo);
      *(bf16x8*)(dst + kh * 256) = hi;
      *(bf16x8*)(dst + kPlaneBlock + kh * 256) = lo;
    }
    return;
  }
  __shared__ float bound[2][16];
  const int ab = tid >> 7;
  const int r = (tid >> 3) & 15;
  const int t = tid & 7;  // inputs 16 t .. + 15: k step t
  const int hid = 16 * (int)blockIdx.x + r;
  const float* src = (ab ? a.w_b : a.w_a) + (int64_t)hid * kChannels + 16 * t;
  float w[16], s2 = 0.f, s1 = 0.f, mw = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 v = *(const f32x4*)(src + 4 * i);
    const float raw[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int in = 16 * t + 4 * i + e;
      const float g = a.ln_w ? a.ln_w[in] : 1.f, b = a.ln_b ? a.ln_b[in] : 0.f;
      const float x = g * raw[e];
      w[4 * i + e] = x;
      s2 = __builtin_fmaf(x, x, s2);
      s1 = __builtin_fmaf(b, raw[e], s1);
      mw = __builtin_elementwise_maximum(mw, __builtin_fabsf(x));
    }
  }
#pragma unroll
  for (int d = 1; d < 8; d <<= 1) {
    s2 += __shfl_xor(s2, d);
    s1 += __shfl_xor(s1, d);
    mw = __builtin_elementwise_maximum(mw, __shfl_xor(mw, d));
  }
  const int e = plane_exp(mw);
  if (t == 0) {
    a.exps[kExpW + ab * kHid + hid] = e;
    a.fbias[ab * kHid + hid] = s1;
    bound[ab][r] = __builtin_sqrtf(128.f * s2) + __builtin_fabsf(s1);
  }
  __bf16* dst = a.planes + (int64_t)(hid >> 5) * kChunkValues +
                ((ab * 8 + t) * 2) * kPlaneBlock + (hid & 31) * 8;
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) {
    bf16x8 hi, lo;
    split_f16(ldexp8(f32x8{w[8 * kh], w[8 * kh + 1], w[8 * kh + 2], w[8 * kh + 3], w[8 * kh + 4],
                           w[8 * kh + 5], w[8 * kh + 6], w[8 * kh + 7]},
                     e),
              hi, lo);
    *(bf16x8*)(dst + kh * 256) = hi;
    *(bf16x8*)(dst + kPlaneBlock + kh * 256) = lo;
  }
  __syncthreads();
  if (tid < 64) {
    const float bh =
        wave_max(tid < 16 ? __builtin_elementwise_maximum(bound[0][tid], 0.2785f) * bound[1][tid]
                          : 0.f);
    if (tid == 0) {
      a.exps[kExpPart + blockIdx.x] = __builtin_bit_cast(int, bh);
      if (blockIdx.x == 0) a.exps[kExpX] = plane_exp(11.3137085f * (1.0f + 0x1p-10f));
    }
  }
}

// Work-groups of 8 waves in three modes; a work-group runs its full tiles and
// then at most one tile of the other two (launch_transition chooses).
//
// Full tiles: work-group g serves row tiles g, g + grid, ... < full_tiles
// (256 rows each, 32 per wave).  Chunk k of the work-group's sequence (chunk
// k % 16 of a tile) sits in LDS stage k % 3; it is copied in two chunks ahead
// (each wave copying 6 KB of it): at chunk k - 2, right after the barrier
// that shows every wave done with chunk k - 3, whose stage it takes.  72 us
// per tile, 1.06 PFLOP/s of executed fp16; without the silu's arithmetic 63,
// without the copies 67.  Neither reading each step's operands a step ahead
// nor running the SIMD's two waves half a chunk apart changed it.
//
// Half tiles (left_rows 128): 128 rows per work-group over the same ring.
// Waves w and w + 4 share 32 rows; wave split s = w / 4 takes hidden channels
// 16 s .. 16 s + 15 of each chunk, value and gate as the two halves of one
// product's rows, so a tile is half the work of a full one on all eight
// waves; the two partial outputs are added through LDS.
//
// Small tiles (left_rows 32 or 64): row group w % R, R = left_rows / 32, is
// served by the 8 / R waves w / R, each passing every (8 / R)-th chunk.  Each
// wave streams its chunks' planes through 16 KB of LDS of its own, four 4 KB
// steps deep, with no barriers; the partial outputs are added through LDS in
// wave order.  Bound by the planes from L2 (each wave reads 2 R chunks of 48 KB:
// 768 R KB per tile).
//
// The rows that do not fill a round of full tiles take the smallest of these
// that one more round covers: at N = 384 the last 64 of 576 tiles as 256
// small tiles 45 us instead of 72, at N = 160 all rows as 200 half tiles 46
// us instead of 66, at N = 64 as 128 small tiles 20 us.
constexpr int kStagesT = 3;
constexpr int kPartBytes = 64 * 64 * 4;  // a wave's partial output
constexpr int kStepBytes = 4096;         // small tiles: planes of one step
__global__ __launch_bounds__(kFusedWaves * 64, 1) void transition_fused_kernel(
    TransitionArgs a, int64_t rows, int64_t full_tiles, int left_rows) {
  __shared__ __attribute__((aligned(16))) uint8_t wbuf[kStagesT][kChunkBytes];
  static_assert(kFusedWaves * kPartBytes <= kStagesT * kChunkBytes, "partials fit the ring");
  static_assert(4 * kStepBytes <= kPartBytes, "a wave's step ring fits its partial output");
  __shared__ __attribute__((aligned(16))) float fb[2][kHid];
  __shared__ __attribute__((aligned(16))) int few[2][kHid];  // -(e_x + e_w) per W' row

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l32 = lane & 31;

  const int64_t my_tiles =
      full_tiles > blockIdx.x ? (full_tiles - 1 - blockIdx.x) / gridDim.x + 1 : 0;
  const int64_t left_row = full_tiles * kFusedRows + (int64_t)blockIdx.x * left_rows;
  const bool has_left = left_rows != 0 && left_row < rows;
  const bool has_half = has_left && left_rows == kFusedRows / 2;
  // chunks this work-group passes through the ring
  const int64_t total = (my_tiles + (has_half ? 1 : 0)) * kChunks;
  constexpr int kWaveBytes = kChunkBytes / kFusedWaves;  // 6 KB
  const uint8_t* const planes = reinterpret_cast<const uint8_t*>(a.planes);
  const uint8_t* csrc = planes + w * kWaveBytes + lane * 16;
  auto dma = [&](int64_t k) {
    const uint8_t* src = csrc + (k % kChunks) * kChunkBytes;
    uint8_t* dst = wbuf[k % kStagesT] + w * kWaveBytes;
#pragma unroll
    for (int i = 0; i < kWaveBytes / 1024; ++i) lds_dma16(src + 1024 * i, dst + 1024 * i);
  };
  if (total > 0) dma(0);
  if (total > 1) dma(1);

  const int ex = __builtin_amdgcn_readfirstlane(a.exps[kExpX]);
  float bh = 0.f;
  for (int g = 0; g < kPrepUp; ++g)
    bh = __builtin_elementwise_maximum(bh, __builtin_bit_cast(float, a.exps[kExpPart + g]));
  // the margin covers the roundings of the bound and of g, v and h
  const int eh = __builtin_amdgcn_readfirstlane(plane_exp(bh * (1.0f + 0x1p-8f)));
  for (int i = tid; i < 2 * kHid; i += kFusedWaves * 64) {
    fb[i / kHid][i % kHid] = a.fbias[i];
    few[i / kHid][i % kHid] = -(ex + a.exps[kExpW + i]);
  }
  // -(e_h + e_o) of this lane's output channels 32 ob + l32
  int eout[4];
#pragma unroll
  for (int ob = 0; ob < 4; ++ob) eout[ob] = -(eh + a.exps[kExpO + 32 * ob + l32]);

  // Operand reads: lane (l32, half) reads row l32's 8 values of k half `half`.
  const uint32_t rd = (uint32_t)(half * 512 + l32 * 16);

  bf16x8 yh[8], yl[8];
  // This lane's row (rows past the end repeat the last row) and its channels
  // 16 t + 8 half + e (the B operand of the up products), normalised.
  auto load_row = [&](int64_t row) {
    const int64_t rr = min(row, rows - 1);
    const int64_t ri = rr / a.rows_j;
    const float* src = a.x + ri * a.xs_i + (rr - ri * a.rows_j) * a.xs_j + 8 * half;
    f32x8 xv[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const f32x4 u = *(const f32x4*)(src + 16 * t);
      const f32x4 v = *(const f32x4*)(src + 16 * t + 4);
      xv[t] = f32x8{u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    }
    // LayerNorm over the row's 128 channels: this lane's 64 and lane l ^ 32's.
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s += xv[t][e];
    }
    const auto ts = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, s),
                                                     __builtin_bit_cast(unsigned, s), false, false);
    const float mean = (__builtin_bit_cast(float, (unsigned)ts[0]) +
                        __builtin_bit_cast(float, (unsigned)ts[1])) * (1.0f / kChannels);
    float q = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      xv[t] = xv[t] - mean;
#pragma unroll
      for (int e = 0; e < 8; ++e) q += xv[t][e] * xv[t][e];
    }
    const auto tq = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, q),
                                                     __builtin_bit_cast(unsigned, q), false, false);
    const float var = (__builtin_bit_cast(float, (unsigned)tq[0]) +
                       __builtin_bit_cast(float, (unsigned)tq[1])) * (1.0f / kChannels);
    const float sc = __builtin_ldexpf(__builtin_amdgcn_rsqf(var + a.eps), ex);
#pragma unroll
    for (int t = 0; t < 8; ++t) split_f16(xv[t] * sc, yh[t], yl[t]);
  };
  // Four values of h = silu(a) * b (scaled by 2^e_h) of this lane's row for
  // hidden channels m .. m + 3, from the products' registers r .. r + 3.
  auto hidden4 = [&](int m, const float* g, const float* v, float* h) {
    const f32x4 ba = *(const f32x4*)&fb[0][m];
    const f32x4 bb = *(const f32x4*)&fb[1][m];
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const i32x4 sa = *(const i32x4*)&few[0][m];
    const i32x4 sb = *(const i32x4*)&few[1][m];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float gg = __builtin_ldexpf(g[e], sa[e]) + ba[e];
      const float vv = __builtin_ldexpf(v[e], sb[e]) + bb[e];
      h[e] = __builtin_ldexpf(gg * sigmoidf_(gg) * vv, eh);
    }
  };
  // A chunk's h from its value and gate products, as planes.
  auto hidden = [&](int c, const f32x16& gacc, const f32x16& vacc, bf16x8 (&hh)[2],
                    bf16x8 (&hl)[2]) {
    float hv[16];
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      const float g[4] = {gacc[4 * qd], gacc[4 * qd + 1], gacc[4 * qd + 2], gacc[4 * qd + 3]};
      const float v[4] = {vacc[4 * qd], vacc[4 * qd + 1], vacc[4 * qd + 2], vacc[4 * qd + 3]};
      hidden4(kChunkHid * c + 8 * qd + 4 * half, g, v, hv + 4 * qd);
    }
#pragma unroll
    for (int st = 0; st < 2; ++st)
      split_f16(f32x8{hv[8 * st + 0], hv[8 * st + 1], hv[8 * st + 2], hv[8 * st + 3],
                      hv[8 * st + 4], hv[8 * st + 5], hv[8 * st + 6], hv[8 * st + 7]},
                hh[st], hl[st]);
  };
  auto up_step = [&](int t, bf16x8 ah, bf16x8 al, bf16x8 bh_, bf16x8 bl, f32x16& gacc,
                     f32x16& vacc) {
    gacc = mfma_f16(ah, yh[t], gacc);
    vacc = mfma_f16(bh_, yh[t], vacc);
    gacc = mfma_f16(ah, yl[t], gacc);
    vacc = mfma_f16(bh_, yl[t], vacc);
    gacc = mfma_f16(al, yh[t], gacc);
    vacc = mfma_f16(bl, yh[t], vacc);
  };
  const bool residual = a.accumulate != 0;
  // out[row][32 ob + l32] of register r of output block ob: row row0 +
  // mfma_row(r, half)
  auto put = [&](int64_t row, int col, float val) {
    if (row >= rows) return;
    const int64_t i = row / a.rows_j;
    float* d = a.out + i * a.os_i + (row - i * a.rows_j) * a.os_j + col;
    *d = residual ? *d + val : val;
  };

  int64_t k = 0;
  // Chunk k of the ring has landed for every wave; starts chunk k + 2.
  auto advance = [&]() -> const uint8_t* {
    // chunk k landed: only chunk k + 1's six copies may still be pending
    if (k + 1 < total)
      wait_vmcnt<6>();
    else
      wait_vmcnt<0>();
    __syncthreads();  // chunk k landed for every wave; chunk k - 1's stage is free
    if (k + 2 < total) dma(k + 2);
    return wbuf[k % kStagesT];
  };
  for (int64_t tile = blockIdx.x; tile < full_tiles; tile += gridDim.x) {
    const int64_t row0 = tile * kFusedRows + 32 * w;
    load_row(row0 + l32);
    f32x16 o[4] = {};
    for (int c = 0; c < kChunks; ++c, ++k) {
      const uint8_t* base = advance() + rd;
      auto blk = [&](int b) -> bf16x8 { return *(const bf16x8*)(base + b * 1024); };
      f32x16 gacc = {}, vacc = {};
#pragma unroll
      for (int t = 0; t < 8; ++t)
        up_step(t, blk(2 * t), blk(2 * t + 1), blk(16 + 2 * t), blk(17 + 2 * t), gacc, vacc);
      bf16x8 hh[2], hl[2];
      hidden(c, gacc, vacc, hh, hl);
#pragma unroll
      for (int ob = 0; ob < 4; ++ob) {
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const int b0 = kUpBlocks + (ob * 2 + st) * 2;
          const bf16x8 wh = blk(b0), wl = blk(b0 + 1);
          o[ob] = mfma_f16(hh[st], wh, o[ob]);
          o[ob] = mfma_f16(hh[st], wl, o[ob]);
          o[ob] = mfma_f16(hl[st], wh, o[ob]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = row0 + mfma_row(r, half);
      if (row >= rows) continue;
      const int64_t i = row / a.rows_j;
      float* d = a.out + i * a.os_i + (row - i * a.rows_j) * a.os_j + l32;
#pragma unroll
      for (int ob = 0; ob < 4; ++ob) {
        const float val = __builtin_ldexpf(o[ob][r], eout[ob]);
        d[32 * ob] = residual ? d[32 * ob] + val : val;
      }
    }
  }

  if (has_half) {
    const int split = w >> 2;
    const int64_t row0 = left_row + 32 * (w & 3);
    load_row(row0 + l32);
    // The up operand's 32 rows: hidden 16 split + l32 % 16 of a (l32 < 16) or
    // of b, whose blocks lie 16 KB further.
    const uint32_t rdu =
        (uint32_t)((l32 >> 4) * 16 * 1024 + half * 512 + (16 * split + (l32 & 15)) * 16);
    f32x16 o[4] = {};
    for (int c = 0; c < kChunks; ++c, ++k) {
      const uint8_t* stage = advance();
      // All operands of a phase are read before its products: a step of
      // three products is shorter than an LDS read.
      bf16x8 u[16];
#pragma unroll
      for (int b = 0; b < 16; ++b) u[b] = *(const bf16x8*)(stage + rdu + b * 1024);
      __builtin_amdgcn_sched_barrier(0);
      f32x16 c0 = {}, c1 = {};
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f32x16& x0 = t & 1 ? c1 : c0;
        f32x16& x1 = t & 1 ? c0 : c1;
        x0 = mfma_f16(u[2 * t], yh[t], x0);
        x1 = mfma_f16(u[2 * t], yl[t], x1);
        x0 = mfma_f16(u[2 * t + 1], yh[t], x0);
      }
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 dn[8];
#pragma unroll
      for (int b = 0; b < 8; ++b)
        dn[b] = *(const bf16x8*)(stage + rd +
                                 (kUpBlocks + ((b >> 1) * 2 + split) * 2 + (b & 1)) * 1024);
      __builtin_amdgcn_sched_barrier(0);
      // registers 0-7: a's rows 8 (r / 4) + 4 half + r % 4, registers 8-15: b's
      const f32x16 x = c0 + c1;
      float hv[8];
#pragma unroll
      for (int qd = 0; qd < 2; ++qd) {
        const float g[4] = {x[4 * qd], x[4 * qd + 1], x[4 * qd + 2], x[4 * qd + 3]};
        const float v[4] = {x[8 + 4 * qd], x[9 + 4 * qd], x[10 + 4 * qd], x[11 + 4 * qd]};
        hidden4(kChunkHid * c + 16 * split + 8 * qd + 4 * half, g, v, hv + 4 * qd);
      }
      bf16x8 hh, hl;
      split_f16(f32x8{hv[0], hv[1], hv[2], hv[3], hv[4], hv[5], hv[6], hv[7]}, hh, hl);
#pragma unroll
      for (int ob = 0; ob < 4; ++ob) {
        o[ob] = mfma_f16(hh, dn[2 * ob], o[ob]);
        o[ob] = mfma_f16(hh, dn[2 * ob + 1], o[ob]);
        o[ob] = mfma_f16(hl, dn[2 * ob], o[ob]);
      }
    }
    // Split 0 stores output blocks 0 and 1, split 1 blocks 2 and 3, each
    // adding the other wave's partial.
    float* const part = reinterpret_cast<float*>(wbuf);
    __syncthreads();  // the ring is free (its last copy landed before the last chunk)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        part[(w * 32 + 16 * i + r) * 64 + lane] = split ? o[i][r] : o[2 + i][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float other = part[((w ^ 4) * 32 + 16 * i + r) * 64 + lane];
        const float sum = split ? other + o[2 + i][r] : o[i][r] + other;
        put(row0 + mfma_row(r, half), 32 * (2 * split + i) + l32,
            __builtin_ldexpf(sum, split ? eout[2 + i] : eout[i]));
      }
    return;
  }
  if (!has_left) return;  // every copy landed before the last chunk

  const int groups = left_rows >> 5;        // R
  const int splits = kFusedWaves / groups;  // waves per row group
  const int group = w % groups;
  const int split = w / groups;
  const int64_t row0 = left_row + 32 * group;
  // The wave's own ring: step q of its sequence (12 per chunk: 8 up steps of
  // a hi, a lo, b hi, b lo, then 4 down steps of one output block) in slot
  // q % 4.
  __syncthreads();  // fb and few are written; the shared ring is free
  uint8_t* const ring = &wbuf[0][0] + w * kPartBytes;
  const int nq = 12 * (kChunks / splits);
  auto step_dma = [&](int q) {
    if (q >= nq) return;
    const int c = split + splits * (q / 12), t = q % 12;
    const uint8_t* src = planes + (int64_t)c * kChunkBytes + lane * 16;
    uint8_t* dst = ring + (q & 3) * kStepBytes;
    // up step t: blocks 2 t, 2 t + 1 of a, then of b (16 blocks further);
    // down step: four consecutive blocks
    const uint8_t* s0 = src + (t < 8 ? 2 * t : kUpBlocks + 4 * (t - 8)) * 1024;
    const uint8_t* s1 = s0 + (t < 8 ? 16 * 1024 : 2 * 1024);
    lds_dma16(s0, dst);
    lds_dma16(s0 + 1024, dst + 1024);
    lds_dma16(s1, dst + 2048);
    lds_dma16(s1 + 1024, dst + 3072);
  };
  load_row(row0 + l32);
#pragma unroll
  for (int q = 0; q < 4; ++q) step_dma(q);
  // Step q's four operands; its slot is then refilled with step q + 4.
  auto step = [&](int q, bf16x8 (&x)[4]) {
    // only steps q + 1 .. q + 3 may still be pending
    if (q + 3 < nq)
      wait_vmcnt<12>();
    else
      wait_vmcnt<0>();
    const uint8_t* at = ring + (q & 3) * kStepBytes + rd;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = *(const bf16x8*)(at + 1024 * i);
    // the reads are done before the copy into their slot starts
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3])::"memory");
    step_dma(q + 4);
  };
  f32x16 o[4] = {};
  for (int c = split, q0 = 0; c < kChunks; c += splits, q0 += 12) {
    f32x16 gacc = {}, vacc = {};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      bf16x8 x[4];
      step(q0 + t, x);
      up_step(t, x[0], x[1], x[2], x[3], gacc, vacc);
    }
    bf16x8 hh[2], hl[2];
    hidden(c, gacc, vacc, hh, hl);
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) {
      bf16x8 x[4];
      step(q0 + 8 + ob, x);
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        o[ob] = mfma_f16(hh[st], x[2 * st], o[ob]);
        o[ob] = mfma_f16(hh[st], x[2 * st + 1], o[ob]);
        o[ob] = mfma_f16(hl[st], x[2 * st], o[ob]);
      }
    }
  }
  float* const part = reinterpret_cast<float*>(&wbuf[0][0]);
#pragma unroll
  for (int ob = 0; ob < 4; ++ob)
#pragma unroll
    for (int r = 0; r < 16; ++r) part[(w * 64 + ob * 16 + r) * 64 + lane] = o[ob][r];
  __syncthreads();
  // wave (split, group) sums and stores its share of the group's values
  const int share = 64 / splits;
  for (int i = split * share; i < (split + 1) * share; ++i) {
    float sum = 0.f;
    for (int p = 0; p < splits; ++p) sum += part[((p * groups + group) * 64 + i) * 64 + lane];
    const int col = 32 * (i >> 4) + l32;
    put(row0 + mfma_row(i & 15, half), col, __builtin_ldexpf(sum, -(eh + a.exps[kExpO + col])));
  }
}

}  // namespace

hipError_t launch_transition(const TransitionArgs& a, hipStream_t stream) {
  const int64_t rows = (int64_t)a.rows_i * a.rows_j;
  if (rows == 0) return hipSuccess;
  if (a.planes == nullptr || a.fbias == nullptr || a.exps == nullptr) return hipErrorInvalidValue;
  const int64_t tiles = (rows + kFusedRows - 1) / kFusedRows;
  if (tiles > 0x7fffffff) return hipErrorInvalidValue;
  // Whole rounds of full tiles over the CUs, then the rows left over as the
  // smallest tiles that one more round covers (32, 64 or 128 rows); a
  // remainder of more than 128 rows per CU runs as full tiles.
  const int64_t cus = device_cu_count();
  int64_t full = tiles / cus * cus;
  const int64_t left = std::max<int64_t>(rows - full * kFusedRows, 0);
  int left_rows = 0;
  if (left > 0) {
    for (int r = 32; r <= kFusedRows / 2 && left_rows == 0; r *= 2)
      if (left <= cus * r) left_rows = r;
    if (left_rows == 0) full = tiles;
  }
  const int64_t units = left_rows ? (left + left_rows - 1) / left_rows : 0;
  const int64_t grid = std::min<int64_t>(std::max(full, units), cus);
  hipError_t e;
  hipLaunchKernelGGL(transition_prep_kernel, dim3(kPrepUp + kPrepDown), dim3(256), 0, stream, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(transition_fused_kernel, dim3((uint32_t)grid), dim3(kFusedWaves * 64), 0,
                     stream, a, rows, full, left_rows);
  return hipGetLastError();
}

}  // namespace fpx
