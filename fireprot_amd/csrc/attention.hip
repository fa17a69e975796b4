// Flash-style triangle attention on the reference C-ABI layout (q, k, v, out
// [B][n][4][32], a shared [4][n][S] bias): the kernel behind ck_attention,
// ck_attention_exact1536, ck_attention_vector_bias1000, fpx_attn_core and
// fpx_attn_core_masked.  The block and the strided (OpenFold3) entries run
// attention_split_kernel on planes staged in a workspace; these entries have
// none, so this kernel splits its operands as it goes.
//
// One work-group = (outer row b, head h, 128 queries); four wavefronts, each
// owning 32 queries.  Keys are streamed in tiles of 32.  Both products run on
// v_mfma_f32_32x32x16_f16 with power-of-two scaled fp16 (hi, lo) planes and
// three terms (FP32 accuracy, split.hpp).  Per tile the four waves load its K
// and V rows two tiles ahead, find the tile's largest |K| and |V| one tile
// ahead, and split them into planes in LDS (double-buffered, one barrier per
// tile), each value once for the work-group's 128 queries:
//   - q by 2^e_q (each wave's 32 queries), K by 2^e_k (each tile);
//   - V by 2^E, E the smallest plane exponent of the tiles so far, so the
//     weights of all tiles enter P.V at one scale; when a tile lowers E, O is
//     scaled by the exact power of two between.
// S^T = K Q^T and O^T += V^T P^T are transposed, so each lane column (lane %
// 32) holds one query in both results: row statistics, the P operand and the
// O rescale live in the lane that needs them, and the only cross-lane step is
// an xor-32 exchange of a tile max.
//
// The bias comes as rows of [n][S]: a wave's 32 x 32 fragment is copied by
// global_load_lds as eight rows of 128 contiguous bytes per instruction into
// 4 KB of LDS of its own and read back in accumulator order.  Loaded straight
// into accumulator order, each instruction touches 32 rows.
//
// Rows with at least one unmasked key (fast): logits fma(acc, 2^-(e_q+e_k),
// bias) in natural units (plus the mask bias where a mask is given), weights
// P' = exp2(fma(x, log2(e), -c)) with one integer reference c per query, 7
// below the ceiling of the largest logit when it was set: no max is formed
// until a lane's 16 weights of a tile sum past 2^15 (or at the first tile).
// A masked key of such a row gets weight exactly 0 whatever the rounding of
// its logit, because its logit is about -1e9 below the row max.
//
// Rows whose keys are all masked (exact): fl(fl(s + mask_bias) + bias) in
// natural units, the native order (patches/protenix/0005-*.patch:36-45;
// kernels/amd/fireprot_softmax_fp32.cpp:33-35).  These logits are quantised to
// the FP32 spacing of -1e9 (64), and this order reproduces which keys tie at
// the max.  Weights are exp2(fma(x, log2 e, -c) - s) with c = fl(m log2 e) of a
// lazy running max m (rescaled when a tile max exceeds it by 2^8) and s = m
// log2(e) - c, so equal logits get equal weights, and the largest is in range
// however far c is rounded (by up to 2^11 at 3e10).
//
// A row whose logits are all -inf gives NaN, as torch.softmax does.  fp16
// planes cannot carry an infinity beside finite values (its residual is NaN),
// so a work-group that meets a non-finite q, k or v computes its rows on the
// FP32 matrix cores (attend_f32) with the native propagation.
//
// Range.  A plane pair resolves 2^-25 in scaled units, 2^-39 of the largest
// value it is scaled with, whereas FP32 keeps 24 bits of every value.  A
// work-group whose operands need more runs on attend_f32 as well:
//   - logits: what the planes drop of one logit is at most 32 products of one
//     operand's largest value and the other's resolution, for both operands:
//     64 2^-39 max|q| max|K| = 2^-33 max|q| max|K|.  Up to max|q| max|K| =
//     2^10 (kMaxProduct) that is 2^-23, the rounding of a logit near 1.  Past
//     it the planes stay when no nonzero row and no nonzero channel of the
//     wave's q or of the tile's K lies below 2^-8 of the largest value
//     (kEvenShare): then they drop at most 2^-39 sqrt(32) 2 2^8 |q|_2 |k|_2 =
//     2^-27.5 |q|_2 |k|_2, less than FP32 sums round.
//   - V, looked at when the sums are complete, in scaled units (max|V| in
//     [2^14, 2^15)): what the planes drop of O' = sum P' V' is at most
//     2^-25 l' (V's resolution) and about 2^-25 2^14 sqrt(N / 3) (that of the
//     weights, uniformly distributed errors of random sign).  A query whose
//     largest |O'| over the channels is not 2^22 times that sum (kRowShare,
//     kWeightShare) gets its weight from keys of V far below the largest (a
//     masked key's, say): FP32.  (Equal weights round alike and their errors
//     add up, N / sqrt(N / 3) times as much; so do the roundings of an FP32
//     sum of N like terms, and the latter are the larger wherever |O'| passes
//     2^14, as it does here from N = 192 on.)  Likewise FP32 when some
//     channel's largest |V| is nonzero and below 1, 2^-14 or less of all: its
//     error would pass 2^-25 of it.
// Tiles of V further apart than 2^20 (kMaxSpread; padded keys holding anything
// are the usual cause) go to FP32 as they are met.  So the planes' error is
// relative to the largest output of the row and to the largest V of the
// channel.  The looks cost 1.6% at N = 1536 (3080 to 3129 us; 3 to 4% with a
// mask: B = 64 508 to 525 us where every key is masked) and at most 0.6 us of 13
// at N = 128.  attend_f32 runs at the rate of a kernel of its own
// (B = 64, N = 1536: 786 us for a NaN in the first tile, 406 on the planes); a
// value or range that only the last tiles or the sums show costs both, 1.2 ms.
//
// Bound: VALU issue beside the matrix cores (236 VALU instructions and 12 MFMAs
// per wave and tile; VALU 86% busy, matrix cores 31%).  At B = 512, N = 1536: 3.13 ms; on the FP32
// matrix cores, which never overlap with VALU work, 5.39 ms.  N = 384 176 us
// against 304.
#include "attn_common.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "split.hpp"

#include <cmath>
#include <type_traits>

namespace fpx {
namespace {

constexpr int kThreads = 256;
constexpr int kPlaneBytes = 2048;              // 32 rows of 64 bytes
constexpr int kTileBytes = 4 * kPlaneBytes;    // K hi, K lo, V^T hi, V^T lo
constexpr int kBiasBytes = 32 * kBk * 4;       // a wave's bias fragment
constexpr float kPlaneMax = 32768.0f;          // bound on a lane's 16 scaled weights
// Weights enter P.V as up to 2^7 and more.  2^10 would resolve small ones eight times finer and
// keep more rows off attend_f32, but moves the reference more often: 2 to 4% at logits of 4
// standard deviations.
constexpr float kShift = 7.0f;
constexpr int64_t kMaxBiasStride = 1 << 25;    // 31 rows within 32-bit byte offsets
constexpr float kBigLogit = 4194304.0f;        // 2^22: past it, references take no shift
// Range of the planes (file comment).
constexpr float kMaxProduct = 1024.0f;
constexpr float kEvenShare = 0x1p-8f;
constexpr float kRowShare = 0.125f;      // 2^22 2^-25
constexpr float kWeightShare = 1182.4f;  // 2^22 2^-25 2^14 / sqrt(3)
constexpr int kMaxSpread = 20;
constexpr int kNoExp = 141;  // V's exponent while every tile was zero

// The planes' ring and bias fragments; attend_f32's K and V tiles in their place.
constexpr int kPad = 4;  // LDS row padding (floats): conflict-free b128 reads
typedef float KTile[kBk][kHeadDim + kPad];  // [key][channel]
typedef float VTile[kHeadDim][kBk + kPad];  // [channel][key]
constexpr int kPoolBytes = 2 * kTileBytes + kThreads / 64 * kBiasBytes;
static_assert(2 * sizeof(KTile) + 2 * sizeof(VTile) <= kPoolBytes, "FP32 tiles fit the pool");

// v_mfma_f32_32x32x2_f32: A[row][k] in lane row + 32 k, B[k][col] in lane col + 32 k,
// result in the 32x32 layout (common.hpp).
__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// The work-group's rows on the FP32 matrix cores, for operands that the planes
// do not hold, and for bias rows so far apart that a wave's 32 span more than
// 4 GB.  K and V^T tiles are staged in `pool` (double buffers, one
// barrier per tile), each a tile ahead in registers; the bias is loaded a tile
// ahead into the registers its logits take.  On gfx950 an FP32 MFMA and VALU
// work never overlap, so each tile runs S^T, softmax and O^T += V^T P^T in
// order.  Logits, reference and weights are those of the planes' path, with
// the reference snapped to 0 while the row's largest logit lies within kSnap,
// and moved when the running sum passes kSumLimit.
__device__ __forceinline__ void attend_f32(const AttnArgs& a, int b, int h, int jq, int nkt,
                                           uint8_t* pool) {
  KTile* const Ks = reinterpret_cast<KTile*>(pool);
  VTile* const Vs = reinterpret_cast<VTile*>(pool + 2 * sizeof(KTile));
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int half = lane >> 5;
  const int l32 = lane & 31;
  const int row8 = tid >> 3;         // key of the thread's K and V loads
  const int col4 = (tid & 7) * 4;    // and their channels
  const int last = nkt - 1;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const int64_t head = ((int64_t)b * a.n * kHeads + h) * kHeadDim;

  int found = a.mbias == nullptr;
  if (!found) {
    for (int k = tid; k < a.n; k += kThreads) found |= a.mbias[(int64_t)b * a.mb_stride + k] == 0.0f;
  }
  // the barrier also releases the pool
  const bool has_unmasked = __syncthreads_or(found) != 0;

  auto rows = [&](const float* base, int t) -> f32x4 {
    const int key = t * kBk + row8;
    return key < a.n ? *(const f32x4*)(base + head + (int64_t)key * kHidden + col4) : zero;
  };
  auto put = [&](int stage, f32x4 k, f32x4 v) {
    *(f32x4*)&Ks[stage][row8][col4] = k;
    Vs[stage][col4 + 0][row8] = v.x;
    Vs[stage][col4 + 1][row8] = v.y;
    Vs[stage][col4 + 2][row8] = v.z;
    Vs[stage][col4 + 3][row8] = v.w;
  };
  const bool ok = jq < a.n;
  const float* const brow = a.bias + ((int64_t)h * a.bias_rows + (ok ? jq : 0)) * a.bias_stride;
  auto bias = [&](int t) -> f32x16 {
    f32x4 x[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int key = t * kBk + 8 * rr + 4 * half;  // n % 4 == 0: all four in or out
      x[rr] = ok && key < a.n ? *(const f32x4*)(brow + key) : zero;
    }
    return cat4(x[0], x[1], x[2], x[3]);
  };

  // Q, the B operand of S^T = K Q^T: lane holds Q[jq][16 half + s].
  float qf[16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 v =
        ok ? *(const f32x4*)(a.q + head + (int64_t)jq * kHidden + 16 * half + 4 * i) : zero;
    qf[4 * i + 0] = v.x;
    qf[4 * i + 1] = v.y;
    qf[4 * i + 2] = v.z;
    qf[4 * i + 3] = v.w;
  }

  f32x16 o = {};
  float l_run = 0.f;
  auto run = [&](auto exact_tag) {
    constexpr bool kExact = decltype(exact_tag)::value;
    float m_ref = -INFINITY;  // largest tile max when the reference was last looked at
    float c_ref = 0.f;        // the reference, in log2 units
    float s_ref = 0.f;        // exact path: m_ref log2(e) - c_ref, what c_ref's rounding left
    bool has_ref = false;     // uniform per wave, as big
    bool big = false;
    // As in the planes' path, fast rows round logits past 2^22 (big) to log2
    // units before the reference is taken off.
    auto weights = [&](f32x16& x) {
      if (big) {
#pragma clang fp contract(off)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float y = x[r] * kLog2e;
          x[r] = exp2_fast(y - c_ref);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = exp2_fast(__builtin_fmaf(x[r], kLog2e, -c_ref));
      }
    };
    auto rescale = [&](float alpha) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] *= alpha;
      l_run *= alpha;
    };
    // Logits x in natural units -> weights, in place.
    auto softmax = [&](f32x16& x) {
      if (kExact) {
        const float mt = xor32_max(max16(x));
        if (__any(mt > m_ref + kRescaleNat)) {
          const float m_new = __builtin_elementwise_maximum(m_ref, mt);
          const float c_new = m_new == -INFINITY ? 0.f : m_new * kLog2e;
          rescale(m_ref == -INFINITY ? 0.f : exp2_fast((m_ref - m_new) * kLog2e));
          m_ref = m_new;
          c_ref = c_new;
          s_ref = m_new == -INFINITY ? 0.f : __builtin_fmaf(m_new, kLog2e, -c_new);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r)
          x[r] = exp2_fast(__builtin_fmaf(x[r], kLog2e, -c_ref) - s_ref);
        l_run += sum16(x);
        return;
      }
      float ovf = 0.f;
      if (has_ref) {
        f32x16 p = x;
        weights(p);
        const float l_new = l_run + sum16(p);
        const bool over = !(l_new <= kSumLimit);  // NaN or inf count as overflow
        if (!__any(over)) {
          l_run = l_new;
          x = p;
          return;
        }
        ovf = over ? 1.f : 0.f;
      }
      // Rare, taken by the whole wavefront.  A lane moves its reference only
      // when it has none yet, when its own running sum overflowed, or when
      // this tile's max lies more than kSnap above the reference; the decision
      // is shared by the lane pair (l, l ^ 32) that holds the query.  After a
      // sum overflow the true row max is at least c_ref + 52, so the reference
      // moves up by at least kLift and the weights stay below 2^24.
      const float mt = xor32_max(max16(x)) * kLog2e;
      const bool fresh = m_ref == -INFINITY;
      const bool need = fresh || xor32_max(ovf) > 0.f || mt > c_ref + kSnap;
      m_ref = __builtin_elementwise_maximum(m_ref, mt);
      const float snapped =
          (m_ref == -INFINITY || (m_ref >= -kSnap && m_ref <= kSnap)) ? 0.f : m_ref;
      const float c_new = fresh ? snapped
                          : need ? __builtin_elementwise_maximum(snapped, c_ref + kLift)
                                 : c_ref;
      rescale(fresh ? 0.f : exp2_fast(c_ref - c_new));  // 1 when unchanged
      c_ref = c_new;
      has_ref = __all(m_ref != -INFINITY);
      big = __any(!(__builtin_fabsf(c_ref) < kBigLogit));
      weights(x);
      l_run += sum16(x);
    };

    f32x16 x = bias(0);
    put(0, rows(a.k, 0), rows(a.v, 0));
    f32x4 kx = rows(a.k, min(1, last)), vx = rows(a.v, min(1, last));
    __syncthreads();
    for (int t = 0; t <= last; ++t) {
      const int par = t & 1;
      f32x16 s = {};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 kv = *(const f32x4*)&Ks[par][l32][16 * half + 4 * i];
        s = mfma_f32(kv.x, qf[4 * i + 0], s);
        s = mfma_f32(kv.y, qf[4 * i + 1], s);
        s = mfma_f32(kv.z, qf[4 * i + 2], s);
        s = mfma_f32(kv.w, qf[4 * i + 3], s);
      }
      if (a.mbias != nullptr || (t + 1) * kBk > a.n) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = t * kBk + mfma_row(r, half);
          const float m =
              key < a.n ? (a.mbias ? a.mbias[(int64_t)b * a.mb_stride + key] : 0.f) : -INFINITY;
          s[r] = (s[r] + m) + x[r];  // the native order
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] += x[r];
      }
      x = bias(min(t + 1, last));
      softmax(s);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const f32x4 vv = *(const f32x4*)&Vs[par][l32][8 * rr + 4 * half];
        o = mfma_f32(vv.x, s[4 * rr + 0], o);
        o = mfma_f32(vv.y, s[4 * rr + 1], o);
        o = mfma_f32(vv.z, s[4 * rr + 2], o);
        o = mfma_f32(vv.w, s[4 * rr + 3], o);
      }
      put(par ^ 1, kx, vx);  // the stage every wave left behind at the last barrier
      kx = rows(a.k, min(t + 2, last));
      vx = rows(a.v, min(t + 2, last));
      __syncthreads();
    }
  };
  if (has_unmasked)
    run(std::false_type{});
  else
    run(std::true_type{});

  const float l_tot = xor32_sum(l_run);
  if (!ok) return;
#pragma unroll
  for (int rr = 0; rr < 4; ++rr)
    *(f32x4*)(a.out + head + (int64_t)jq * kHidden + 8 * rr + 4 * half) =
        f32x4{o[4 * rr + 0] / l_tot, o[4 * rr + 1] / l_tot, o[4 * rr + 2] / l_tot,
              o[4 * rr + 3] / l_tot};
}

__global__ __launch_bounds__(kThreads, 4) void attention_kernel(AttnArgs a, int nqt, int nkt,
                                                                uint32_t total, int ppg) {
  __shared__ __attribute__((aligned(16))) uint8_t pool[kPoolBytes];
  uint8_t (*const kv)[kTileBytes] = reinterpret_cast<uint8_t (*)[kTileBytes]>(pool);
  uint8_t (*const bias_lds)[kBiasBytes] =
      reinterpret_cast<uint8_t (*)[kBiasBytes]>(pool + 2 * kTileBytes);
  // each wave's largest |K| and |V| of tile t at [t & 1]; [2]: its largest |q|, and look's answer
  __shared__ float red[3][kThreads / 64][2];
  // largest |V| so far (float bits) of channel l32, a cell for each lane half at the
  // plane reads' offsets, whose address register it shares
  __shared__ __attribute__((aligned(16))) uint8_t channels[kPlaneBytes];
  __shared__ uint32_t low_rows;  // some query's output is below its share

  int b, h, qt;
  attn_item(blockIdx.x, total, a.batch, nqt, ppg, b, h, qt);
  if (b >= a.batch) return;  // padding of the last row group; uniform per work-group
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l32 = lane & 31;
  const int j0 = qt * kBq + 32 * w;
  const int jq = j0 + l32;
  const int last = nkt - 1;

  // The planes' path; false (uniform) when the rows need attend_f32.
  auto attend = [&]() -> bool {
    if (a.bias_stride > kMaxBiasStride) return false;
    const uint32_t rd0 = l32 * 64 + 16 * (half ^ swz(l32));
    auto channel_max = [&]() { return reinterpret_cast<uint32_t*>(channels + rd0); };
    if (w == 0) *channel_max() = 0u;
    if (tid == 0) low_rows = 0u;

    // Row classification.  masked(t): the mask bias is added to tile t's logits
    // (every tile where a mask is given, zeros or not; the tile that ends past
    // n).  has_unmasked: some key k < n of the row has a zero mask bias.
    int found = a.mbias == nullptr;
    if (!found) {
      for (int k = tid; k < a.n; k += kThreads) found |= a.mbias[(int64_t)b * a.mb_stride + k] == 0.0f;
    }
    const bool has_unmasked = __syncthreads_or(found) != 0;
    auto masked = [&](int t) -> bool { return a.mbias != nullptr || (t + 1) * kBk > a.n; };
    // f(r, mask bias of register r's key) over a tile, four registers at a time
    // (all sixteen values at once would not fit the register budget).
    auto with_mask = [&](int t, auto&& f) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        float m[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = t * kBk + 8 * rr + 4 * half + e;
          m[e] = key < a.n ? (a.mbias ? a.mbias[(int64_t)b * a.mb_stride + key] : 0.f) : -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) f(4 * rr + e, m[e]);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    // K rows: thread (key tid / 8, channels 4 (tid % 8) .. + 3).  V: thread
    // (channel tid % 32, keys 4 (tid / 32) .. + 3), so its four keys are
    // adjacent in the V^T planes.  Keys past n are loaded from the last key
    // (no branch around the loads) and zeroed.
    const int kkey = tid >> 3, kc4 = (tid & 7) * 4;
    const int vc = tid & 31, vg = tid >> 5;
    const float* const krow = a.k + ((int64_t)b * a.n * kHeads + h) * kHeadDim;
    const float* const vrow = a.v + ((int64_t)b * a.n * kHeads + h) * kHeadDim;
    auto load_kv = [&](int t, f32x4& kx, f32x4& vx) {
      const int key = t * kBk + kkey;
      kx = *(const f32x4*)(krow + (uint32_t)(min(key, a.n - 1) * kHidden + kc4));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        vx[i] = vrow[(uint32_t)(min(t * kBk + 4 * vg + i, a.n - 1) * kHidden + vc)];
    };
    auto clip_kv = [&](int t, f32x4& kx, f32x4& vx) {  // uniform branch: the last tile at most
      if ((t + 1) * kBk <= a.n) return;
      if (t * kBk + kkey >= a.n) kx = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (t * kBk + 4 * vg + i >= a.n) vx[i] = 0.f;
    };
    auto max4 = [](const f32x4& x) -> float {
      return __builtin_elementwise_maximum(
          __builtin_elementwise_maximum(__builtin_fabsf(x.x), __builtin_fabsf(x.y)),
          __builtin_elementwise_maximum(__builtin_fabsf(x.z), __builtin_fabsf(x.w)));
    };
    float q_max;  // the work-group's largest |q|
    auto note_max = [&](const f32x4& kx, const f32x4& vx, int slot) {
      const float v4 = max4(vx);  // four keys of channel vc
      __hip_atomic_fetch_max(channel_max(), __builtin_bit_cast(uint32_t, v4), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
      const float mk = wave_max(max4(kx)), mv = wave_max(v4);
      if (lane == 0) {
        red[slot][w][0] = mk;
        red[slot][w][1] = mv;
      }
    };
    auto read_max = [&](int slot, float& mk, float& mv) {
      mk = red[slot][0][0];
      mv = red[slot][0][1];
#pragma unroll
      for (int i = 1; i < kThreads / 64; ++i) {
        mk = __builtin_elementwise_maximum(mk, red[slot][i][0]);
        mv = __builtin_elementwise_maximum(mv, red[slot][i][1]);
      }
    };
    // Q planes (B operand of S^T = K Q^T): lane holds Q[jq][16 m + 8 half + e].
    bf16x8 qh[2], ql[2];
    int eq, ek, ev;  // plane exponents of the wave's q, of the tile's K, and E
    // Whether no row or channel of the wave's q (its hi plane) lies below
    // kEvenShare of its largest value, and no nonzero row or channel of K, over
    // the eight keys of the tile (kx, largest |K| mk) that the wave holds.
    auto q_even = [&]() -> bool {
      f16x8 x[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        f32x4 bits = __builtin_bit_cast(f32x4, qh[m]);
        asm volatile("" : "+v"(bits));  // formed here, not ahead of the loop in registers it needs
        x[m] = __builtin_bit_cast(f16x8, bits);
      }
      auto at = [&](int i) { return __builtin_fabsf((float)x[i >> 3][i & 7]); };
      float row = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) row = __builtin_elementwise_maximum(row, at(i));
      row = xor32_max(row);
      const float least = kEvenShare * wave_max(row);
      bool bad = row < least;
#pragma unroll
      for (int i = 0; i < 16; ++i) bad |= half_max(at(i)) < least;
      return !__any(bad);
    };
    auto k_even = [&](const f32x4& kx, float mk) -> bool {
      const float least = kEvenShare * mk;
      float row = max4(kx);
      row = __builtin_elementwise_maximum(row, dpp<0xB1>(row));
      row = __builtin_elementwise_maximum(row, dpp<0x4E>(row));
      row = __builtin_elementwise_maximum(row, dpp<0x141>(row));
      bool bad = row != 0.f && row < least;
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // lanes of equal lane % 8: row_ror:8, row and half swaps
        float c = __builtin_fabsf(kx[e]);
        c = __builtin_elementwise_maximum(c, dpp<0x128>(c));
        const auto r = __builtin_amdgcn_permlane16_swap(
            __builtin_bit_cast(unsigned, c), __builtin_bit_cast(unsigned, c), false, false);
        c = xor32_max(__builtin_elementwise_maximum(__builtin_bit_cast(float, (unsigned)r[0]),
                                                    __builtin_bit_cast(float, (unsigned)r[1])));
        bad |= c != 0.f && c < least;
      }
      return !__any(bad);
    };
    // Whether a tile of these maxima needs no look at its values (false for NaN),
    // and whether one that does fits the planes.  Uniform.
    auto plain = [&](float mk, float mv) { return (q_max * mk <= kMaxProduct) & (mv < INFINITY); };
    int q_known = -1;  // q_even() once it was needed; uniform per wave
    auto look = [&](const f32x4& kx, float mk, float mv) -> bool {
      if (!(mk < INFINITY && mv < INFINITY && q_max * mk <= 0x1p96f)) return false;
      if (q_known < 0) q_known = __builtin_amdgcn_readfirstlane(q_even());
      const bool even = k_even(kx, mk) && q_known != 0;
      // every wave's answer; a barrier ends the iteration before the next look
      if (lane == 0) red[2][w][1] = even ? 0.f : 1.f;
      __syncthreads();
      float bad = 0.f;
#pragma unroll
      for (int i = 0; i < kThreads / 64; ++i) bad += red[2][i][1];
      return bad == 0.f;
    };
    // A staged tile into planes: 16-byte chunk c of a plane's row r sits at
    // chunk c ^ swz(r).  V^T keys lie in the order of the S^T accumulator
    // registers: key group g of four at position 16 (g / 4) + 4 (0, 2, 1,
    // 3)[g % 4].
    const uint32_t kput = kkey * 64 + 16 * ((kc4 >> 3) ^ swz(kkey)) + (kc4 & 4) * 2;
    auto put = [&](int stage, const f32x4& kx, const f32x4& vx, int ek, int ev) {
      bf16x4 hi, lo;
      split_f16(ldexp4(kx, ek), hi, lo);
      *(bf16x4*)(kv[stage] + kput) = hi;
      *(bf16x4*)(kv[stage] + kPlaneBytes + kput) = lo;
      split_f16(ldexp4(vx, ev), hi, lo);
      // vg = 2 w + half: its four keys start at position 16 (w / 2) + 8 half +
      // 4 (w % 2), half w % 2 of the chunk that plane_rd(.., m = w / 2) reads.
      // Formed from that offset here: there is no register to hold it.
      uint32_t flip = 32u * (w >> 1);
      asm volatile("" : "+s"(flip));
      const uint32_t vput = (rd0 ^ flip) + 8 * (w & 1);
      *(bf16x4*)(kv[stage] + 2 * kPlaneBytes + vput) = hi;
      *(bf16x4*)(kv[stage] + 3 * kPlaneBytes + vput) = lo;
    };
    // V's exponent of a tile; a zero tile keeps the one so far
    auto value_exp = [](float m, int so_far) -> int {
      return __builtin_amdgcn_readfirstlane(m == 0.f ? so_far : plane_exp(m));
    };
    auto plane_rd = [&](int stage, int plane, int m) -> bf16x8 {
      return *(const bf16x8*)(kv[stage] + plane * kPlaneBytes + (rd0 ^ (32 * m)));
    };

    // Bias fragment of tile t: instruction i copies rows 8 i + lane / 8 of the
    // wave's 32 queries, 16-byte chunk lane % 8 from that row's chunk
    // (lane % 8) ^ (lane / 8), so the reads in accumulator order are spread over
    // the banks.  Rows past n are row n - 1, keys past n the row's last four:
    // their queries are dropped, their logits masked.
    const int chunk = (lane & 7) ^ (lane >> 3);
    const int jw = min(j0, a.n - 1);  // the wave's first row
    const uint64_t bits =
        (uint64_t)(a.bias + ((int64_t)h * a.bias_rows + jw) * a.bias_stride);
    const uint8_t* const brow = reinterpret_cast<const uint8_t*>(
        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(bits >> 32)) << 32) |
        (uint32_t)__builtin_amdgcn_readfirstlane((int)bits));
    const uint32_t step = 8u * (uint32_t)a.bias_stride * 4u;
    const int rows_left = a.n - 1 - jw;
    const uint32_t bias_at = __builtin_amdgcn_readfirstlane((int)lds_address(bias_lds[w]));
    auto bias_dma = [&](int t) {
      const uint32_t col = 4u * (uint32_t)min(4 * chunk, a.n - 4 - t * kBk);
      const uint8_t* base = brow + (int64_t)t * kBk * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t row = (uint32_t)min(8 * i + (lane >> 3), rows_left);
        lds_dma16_s(row * (step >> 3) + col, base, bias_at + 1024 * i);
      }
    };
    auto bias_rd = [&]() -> f32x16 {
      const uint8_t* src = bias_lds[w] + l32 * 128;
      f32x4 x[4];
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) x[rr] = *(const f32x4*)(src + 16 * ((2 * rr + half) ^ (l32 & 7)));
      return cat4(x[0], x[1], x[2], x[3]);
    };

    f32x4 ka, va;
    {
      const float* src = a.q + (((int64_t)b * a.n + min(jq, a.n - 1)) * kHeads + h) * kHeadDim + 8 * half;
      f32x4 x[4];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        x[2 * m] = *(const f32x4*)(src + 16 * m);
        x[2 * m + 1] = *(const f32x4*)(src + 16 * m + 4);
      }
      f32x4 k0, v0;
      load_kv(0, k0, v0);
      load_kv(last < 1 ? last : 1, ka, va);
      bias_dma(0);
      float mq = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) mq = __builtin_elementwise_maximum(mq, max4(x[i]));
      mq = wave_max(mq);
      eq = __builtin_amdgcn_readfirstlane(plane_exp(mq));
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const f32x4 u = ldexp4(x[2 * m], eq), v = ldexp4(x[2 * m + 1], eq);
        split_f16(f32x8{u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w}, qh[m], ql[m]);
      }
      clip_kv(0, k0, v0);
      clip_kv(last < 1 ? last : 1, ka, va);
      note_max(k0, v0, 0);
      note_max(ka, va, 1);
      if (lane == 0) red[2][w][0] = mq;
      __syncthreads();
      float mk, mv;
      read_max(0, mk, mv);
      q_max = red[2][0][0];
#pragma unroll
      for (int i = 1; i < kThreads / 64; ++i)
        q_max = __builtin_elementwise_maximum(q_max, red[2][i][0]);
      q_max = __builtin_bit_cast(
          float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, q_max)));
      q_max = __builtin_bit_cast(
          float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, q_max)));
      if (!plain(mk, mv) && !look(k0, mk, mv)) {
        wait_vmcnt<0>();  // no copy in flight when the LDS is released
        return false;
      }
      ek = __builtin_amdgcn_readfirstlane(plane_exp(mk));
      ev = value_exp(mv, kNoExp);
      put(0, k0, v0, ek, ev);
      __syncthreads();
    }

    f32x16 o = {};
    float l_run = 0.f;
    bool fits = true;  // uniform
    auto run = [&](auto exact_tag) {
      constexpr bool kExact = decltype(exact_tag)::value;
      const f32x16 zero16 = {};
      // Reference state of this lane's query: m_ref the largest tile max seen
      // when the reference was last looked at (-inf: none yet).
      float m_ref = -INFINITY;
      float c_ref = 0.f;
      float s_ref = -kShift;  // exact path: m_ref log2(e) - c_ref, what its rounding left, - shift
      bool has_ref = false;  // uniform per wave, as big
      bool big = false;
      // Logits x in natural units -> the weights' planes.
      auto softmax = [&](const f32x16& x, bf16x8 (&ph)[2], bf16x8 (&pl)[2]) {
        f32x16 p;
        if (kExact) {
          const float mt = xor32_max(max16(x));
          if (__any(mt > m_ref + kRescaleNat)) {
            const float m_new = __builtin_elementwise_maximum(m_ref, mt);
            const float c_new = m_new == -INFINITY ? 0.f : m_new * kLog2e;
            const float alpha = m_ref == -INFINITY ? 0.f : exp2_fast((m_ref - m_new) * kLog2e);
#pragma unroll
            for (int r = 0; r < 16; ++r) o[r] *= alpha;
            l_run *= alpha;
            m_ref = m_new;
            c_ref = c_new;
            s_ref = (m_new == -INFINITY ? 0.f : __builtin_fmaf(m_new, kLog2e, -c_new)) - kShift;
          }
          // The weights are at most 2^8; the planes and the sum hold them times 2^kShift.
#pragma unroll
          for (int r = 0; r < 16; ++r)
            p[r] = exp2_fast(__builtin_fmaf(x[r], kLog2e, -c_ref) - s_ref);
          l_run += sum16(p);
        } else {
          // Logits past 2^22 (big) are rounded to log2 units before the
          // reference is taken off, so that none exceeds its own maximum.
          auto weights = [&]() {
            if (big) {
#pragma clang fp contract(off)
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const float y = x[r] * kLog2e;
                p[r] = exp2_fast(y - c_ref);
              }
            } else {
#pragma unroll
              for (int r = 0; r < 16; ++r) p[r] = exp2_fast(__builtin_fmaf(x[r], kLog2e, -c_ref));
            }
          };
          weights();
          float ps = sum16(p);
          if (!has_ref || __any(!(ps <= kPlaneMax))) {
            // Rare, taken by the whole wavefront: the first tile, or a tile
            // whose weights would leave the fp16 range.  The reference moves
            // up to kShift below the tile's max rounded up to an integer; the
            // previous sums scale by the exact power of two alpha.  A query
            // whose logits are all -inf so far keeps no reference.
            const float mt = xor32_max(max16(x)) * kLog2e;
            const bool fresh = m_ref == -INFINITY;
            m_ref = __builtin_elementwise_maximum(m_ref, mt);
            const float top = __builtin_ceilf(mt);
            const float to = __builtin_fabsf(top) < kBigLogit ? top - kShift : top;
            const float c_new = fresh ? (m_ref == -INFINITY ? 0.f : to)
                                      : __builtin_elementwise_maximum(c_ref, to);
            const float alpha = fresh ? 0.f : exp2_fast(c_ref - c_new);  // 1 when unchanged
#pragma unroll
            for (int r = 0; r < 16; ++r) o[r] *= alpha;
            l_run *= alpha;
            c_ref = c_new;
            has_ref = __all(m_ref != -INFINITY);
            big = __any(!(__builtin_fabsf(c_ref) < kBigLogit));
            weights();
            ps = sum16(p);
          }
          l_run += ps;
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const f32x8 v = {p[8 * m + 0], p[8 * m + 1], p[8 * m + 2], p[8 * m + 3],
                           p[8 * m + 4], p[8 * m + 5], p[8 * m + 6], p[8 * m + 7]};
          split_f16(v, ph[m], pl[m]);
        }
      };

      for (int t = 0; t <= last; ++t) {
        const int par = t & 1;
        const int e = eq + ek;  // of tile t
        // Tile t + 1 into the other stage, which every wave left behind at the
        // last barrier; then tile t + 2's rows on their way (clamped to the
        // last tile).
        int e_new = ev;
        if (t < last) {
          float mk, mv;
          read_max(par ^ 1, mk, mv);
          const int et = value_exp(mv, ev);
          const bool near = (unsigned)(et - ev + kMaxSpread) <= 2u * kMaxSpread;
          if (__builtin_expect(!(near & plain(mk, mv)), 0)) {
            fits = (near || ev == kNoExp) && (plain(mk, mv) || look(ka, mk, mv));
            if (!fits) break;
          }
          ek = __builtin_amdgcn_readfirstlane(plane_exp(mk));
          e_new = min(ev, et);
          put(par ^ 1, ka, va, ek, e_new);
        }
        load_kv(t + 2 <= last ? t + 2 : last, ka, va);
        asm volatile("" ::: "memory");  // issued here: the wait below counts them
        __builtin_amdgcn_sched_barrier(0);
        f32x16 acc = zero16;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const bf16x8 kh = plane_rd(par, 0, m);
          const bf16x8 kl = plane_rd(par, 1, m);
          acc = mfma_f16(kl, qh[m], acc);
          acc = mfma_f16(kh, ql[m], acc);
          acc = mfma_f16(kh, qh[m], acc);
        }
        // The wave's bias fragment has landed once at most the five row loads
        // above, issued after it, are outstanding.  When nothing reads those
        // rows the compiler may drop the loads: wait for all.
        if (t + 2 <= last)
          wait_vmcnt<5>();
        else
          wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        f32x16 x = bias_rd();
        const float st = __builtin_ldexpf(1.0f, -min(max(e, -126), 126));
        if (kExact) {
          with_mask(t, [&](int r, float m) { x[r] = ((acc[r] * st) + m) + x[r]; });
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) x[r] = __builtin_fmaf(acc[r], st, x[r]);
          if (masked(t)) with_mask(t, [&](int r, float m) { x[r] += m; });
        }
        bf16x8 ph[2], pl[2];
        softmax(x, ph, pl);
        if (t + 2 <= last) {
          clip_kv(t + 2, ka, va);
          note_max(ka, va, par);  // read in iteration t + 1
        }
        if (t < last) bias_dma(t + 1);  // the fragment's reads are done (softmax used them)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const bf16x8 vh = plane_rd(par, 2, m);
          const bf16x8 vl = plane_rd(par, 3, m);
          o = mfma_f16(vl, ph[m], o);
          o = mfma_f16(vh, pl[m], o);
          o = mfma_f16(vh, ph[m], o);
        }
        if (t < last) {
          if (e_new != ev) {  // uniform: O to the scale of tile t + 1
#pragma unroll
            for (int r = 0; r < 16; ++r) o[r] = __builtin_ldexpf(o[r], e_new - ev);
            ev = e_new;
          }
          __syncthreads();
        }
      }
    };
    if (has_unmasked) {
      run(std::false_type{});
    } else {
      run(std::true_type{});
    }
    wait_vmcnt<0>();  // no copy in flight when the LDS is released
    if (!fits) return false;

    const float l_tot = xor32_sum(l_run);
    if (ev != kNoExp) {  // uniform: V is not all zero
      // The shares of the file comment, decided alike by every wave.
      float top = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) top = __builtin_elementwise_maximum(top, __builtin_fabsf(o[r]));
      top = xor32_max(top);
      const float share =
          __builtin_fmaf(kRowShare, l_tot, kWeightShare * __builtin_sqrtf((float)a.n));
      // a NaN top or l_tot stays; l_tot is 0 where every logit is -inf
      if (jq < a.n && l_tot != 0.f && top < share) low_rows = 1u;
      __syncthreads();
      const float c = xor32_max(__builtin_bit_cast(float, *channel_max()));
      if (low_rows != 0u || __any(c != 0.f && __builtin_ldexpf(c, ev) < 1.0f)) return false;
    }
    if (jq < a.n) {
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int c = 8 * rr + 4 * half;  // channels c..c+3 of head h
        // the mean first: the sum itself may pass the largest float once unscaled
        f32x4 ov = {__builtin_ldexpf(o[4 * rr + 0] / l_tot, -ev),
                    __builtin_ldexpf(o[4 * rr + 1] / l_tot, -ev),
                    __builtin_ldexpf(o[4 * rr + 2] / l_tot, -ev),
                    __builtin_ldexpf(o[4 * rr + 3] / l_tot, -ev)};
        *(f32x4*)(a.out + (((int64_t)b * a.n + jq) * kHeads + h) * kHeadDim + c) = ov;
      }
    }
    return true;
  };
  if (!attend()) attend_f32(a, b, h, jq, nkt, pool);
}

}  // namespace

hipError_t launch_attention(int layout, const AttnArgs& a, hipStream_t stream) {
  if (layout != kAttnHeadLast) return hipErrorInvalidValue;
  const int nqt = (int)(round_up(a.n, kBq) / kBq);
  const int nkt = (int)(round_up(a.n, kBk) / kBk);
  const uint64_t groups = ((uint64_t)a.batch + kRowGroup - 1) / kRowGroup;
  const uint64_t total = groups * kRowGroup * kHeads * nqt;
  if (total == 0) return hipSuccess;
  if (total > 0x7fffffffull) return hipErrorInvalidValue;
  const int ppg = pair_group_size(nqt, (uint64_t)kBq * (uint64_t)a.n * sizeof(float));
  hipLaunchKernelGGL(attention_kernel, dim3((uint32_t)total), dim3(kThreads), 0, stream, a, nqt,
                     nkt, (uint32_t)total, ppg);
  return hipGetLastError();
}

}  // namespace fpx
