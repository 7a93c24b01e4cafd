// skinny.hip — fused dequant + matmul for small batches (a few to 128 rows) on MFMA.
//
// C[m, n] = sum_k A[m, k] * deq(W)[n, k] with fp32 accumulation, for the
// batch sizes between the decode GEMV (M = 1..4) and the prefill GEMM: up to
// 64 rows of f32 activations and 128 of f16 in one pass over the weights.
//
// What bounds it: the weight stream (HBM) at small M, then the issue of the
// code unpacking and the MFMAs and the LDS traffic of both operands, which
// overlap the stream only as far as enough bytes are in flight: an HBM round
// trip takes 2-3 us under load on MI355X, so a CU needs about 100 KB on the
// way for its share of the bandwidth.  Hence both operands go to LDS by
// direct loads that hold no registers, in a ring of S stages of whole chunks
// of K (one barrier per chunk, every load 16 bytes per lane where the row's
// chunk is a multiple of 16 bytes), with nothing else in the loop that waits
// on memory.  The kernels before this one held one chunk (f16: weights and
// activations through registers) or three smaller ones with the activations
// through registers (f32) in flight.
//
// (f16 batches of 65 to 128 rows: a chunk is 64 KB of activations and 9 KB of
// Q4_0 codes, so the ring has two stages only and waits for each.)
//
// Measured on MI355X against them (us per launch, graph replay over rotated
// weights; before -> now; the first line from bench.py, the others one sweep):
//   f16 Q4_0  8192x28672  M = 16 / 32 / 64   56.4 / 61.8 / 69.7 -> 42.2 / 49.7 / 61.2
//   f16 Q8_0  4096x14336  M = 16 / 32 / 64   25.6 / 47.1 / 54.9 -> 19.5 / 21.5 / 26.9
//   f16 Q4_0  4096x4096   M = 16 / 64 / 128  11.3 / 22.3 / 23.5 -> 9.0 / 12.1 / 18.8
//   f32 Q8_0  14336x4096  M = 16 / 32        24.2 / 34.0 -> 22.3 / 28.3
//   f32 Q4_0  4096x4096   M = 16             13.0 -> 10.6
//   f32 Q4_0  2048x2048   M = 16 / 64         9.1 / 16.6 -> 7.5 / 11.0
//
// MFMA v_mfma_f32_16x16x32 (f16 or bf16 operands): A = activations (16 rows
// of M), B = weights (16 rows of N), D[m][n] = sum over 32 k.  Lane l holds
// A row l%16, B (weight) row l%16, both for the eight k values of slot
// s = l/16, and D of weight row l%16, activation rows 4s..4s+3.
//
// f32 activations: each activation x is split into two bf16 parts (x ~ b1 +
// b2: b1 the upper half of x, b2 the remainder rounded, within 2^-16 |x|;
// bf16 has f32's exponent range), B = the integer codes, exact in bf16
// (Q4_0: 128 + n, the nibble placed under bf16 exponent bits 0x43 by one
// byte permute per two codes; Q8_0: the signed code), two chained MFMAs give
// sum_k code*x of one block with exact products and fp32 accumulation, and
// the block scale is applied per block: acc += d * D.  The Q4_0 offset of
// -136 (128 of the bf16 placement and the code's own 8) starts each block's
// chain from sum_k (-136)*x, one extra chain per activation tile that all
// weight tiles share.  Slot s holds k = 4s..4s+3 and 16+4s..16+4s+3 (Q4_0:
// the low and high nibbles of code bytes 4s..4s+3) or 8s..8s+7 (Q8_0).
//
// f16 activations: B = RNE(d*q) in fp16 (the bits of dequant_*_f16),
// accumulated across blocks.  Q8_0 slots as above; Q4_0 takes the two blocks
// of a pair with two MFMAs, slot s the code bytes 8(s%2)..8(s%2)+7 of block
// s/2: their low nibbles are eight consecutive k, and so are their high
// ones, so every activation operand is one 16-byte LDS read (8-byte reads of
// the block-wise order conflicted: 1.1 x the time at 16-64 rows).
//
// Work split: a workgroup of 8 waves covers kBN = 16*T*GN weight rows; GN
// groups of T 16-row tiles, each shared by 8/GN waves that split the blocks
// of a chunk (their sums are added in LDS at the end, in wave order).  K may
// also be split over KG workgroups (last arrival adds the partial tiles in
// order).  T, GN, the LDS budget (158 KB, or 78 KB for two workgroups per
// CU) and KG are chosen per launch by a cost model (sk_cost).
#include <algorithm>
#include <type_traits>

#include "../launch.hpp"
#include "common.hpp"

namespace nfk {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Block bytes, and the code bytes of a lane's slot of 8 elements.
template <class QF> struct SkBlk;
template <> struct SkBlk<Q4_0> {
  static constexpr int kBytes = 18, kSlot = 4;
};
template <> struct SkBlk<Q8_0> {
  static constexpr int kBytes = 34, kSlot = 8;
};

__device__ __forceinline__ half2v sk_h2(uint32_t u) { return __builtin_bit_cast(half2v, u); }
__device__ __forceinline__ uint32_t sk_u2(half2v h) { return __builtin_bit_cast(uint32_t, h); }

// 8 fp16 weights RNE(d*q) (the dequant_*_f16 bits) of 8 code bytes: Q8_0 the
// codes, Q4_0 their low (HI = false) or high nibbles.
template <class QF, bool HI>
__device__ __forceinline__ half8 sk_b_f16(uint32_t qa, uint32_t qb, half2v d2) {
  u32x4 o;
  constexpr bool kQ4 = SkBlk<QF>::kSlot == 4;
  const half2v off = kQ4 ? (HI ? half2v{(half_t)-72.f, (half_t)-72.f} : half2v{(half_t)-1032.f, (half_t)-1032.f})
                         : half2v{(half_t)-1152.f, (half_t)-1152.f};
  const uint32_t ex = kQ4 && HI ? 0x54545454u : 0x64646464u;
  const uint32_t ua = kQ4 ? qa & (HI ? 0xF0F0F0F0u : 0x0F0F0F0Fu) : qa ^ 0x80808080u;
  const uint32_t ub = kQ4 ? qb & (HI ? 0xF0F0F0F0u : 0x0F0F0F0Fu) : qb ^ 0x80808080u;
  o.x = sk_u2((sk_h2(__builtin_amdgcn_perm(ex, ua, 0x04010400u)) + off) * d2);
  o.y = sk_u2((sk_h2(__builtin_amdgcn_perm(ex, ua, 0x04030402u)) + off) * d2);
  o.z = sk_u2((sk_h2(__builtin_amdgcn_perm(ex, ub, 0x04010400u)) + off) * d2);
  o.w = sk_u2((sk_h2(__builtin_amdgcn_perm(ex, ub, 0x04030402u)) + off) * d2);
  return __builtin_bit_cast(half8, o);
}

// B operand, f32 activations: the codes as exact bf16 (Q4_0: 128 + n; Q8_0: the signed code).
template <class QF>
__device__ __forceinline__ bf16x8 sk_b_codes(const uint32_t (&q)[SkBlk<QF>::kSlot / 4]) {
  u32x4 o;
  if constexpr (SkBlk<QF>::kSlot == 4) {
    const uint32_t l = q[0] & 0x0F0F0F0Fu, hi = (q[0] >> 4) & 0x0F0F0F0Fu;
    o.x = __builtin_amdgcn_perm(0x43434343u, l, 0x04010400u);
    o.y = __builtin_amdgcn_perm(0x43434343u, l, 0x04030402u);
    o.z = __builtin_amdgcn_perm(0x43434343u, hi, 0x04010400u);
    o.w = __builtin_amdgcn_perm(0x43434343u, hi, 0x04030402u);
  } else {
    o.x = pack_hi16((float)(int8_t)q[0], (float)(int8_t)(q[0] >> 8));
    o.y = pack_hi16((float)(int8_t)(q[0] >> 16), (float)((int32_t)q[0] >> 24));
    o.z = pack_hi16((float)(int8_t)q[1], (float)(int8_t)(q[1] >> 8));
    o.w = pack_hi16((float)(int8_t)(q[1] >> 16), (float)((int32_t)q[1] >> 24));
  }
  return __builtin_bit_cast(bf16x8, o);
}

// Geometry of a variant: MT 16-row activation tiles, T 16-row weight tiles
// per wave, GN wave groups along N, a unit of K per wave and chunk, BUD KB
// of LDS for the ring.
constexpr int kSkWaves = 8;
template <class QF, typename XT, int MT, int T, int GN, int BUD>
struct SkGeom {
  static constexpr int kGK = kSkWaves / GN;                 // waves splitting a chunk's K
  static constexpr int kBN = 16 * T * GN;                   // weight rows of a workgroup
  static constexpr int kUB = (sizeof(XT) == 2 && SkBlk<QF>::kSlot == 4) ? 2 : 1;  // blocks of a unit
  static constexpr int kCK = 32 * kUB * kGK;           // K of a chunk
  static constexpr int kRB = kCK / 32 * SkBlk<QF>::kBytes;  // bytes of a weight row's chunk
  static constexpr int kUW = kRB % 16 == 0 ? 16 : 4;        // bytes per lane of a weight load
  static constexpr int kUR = kRB / kUW;                     // lane loads per row
  static constexpr int kIW = (kBN * kUR + 63) / 64;         // wave loads of weights per chunk
  static constexpr int kXR = kCK * (int)sizeof(XT) / 16;    // 16-byte units of an activation row's chunk
  static constexpr int kIX = 16 * MT * kXR / 64;            // wave loads of activations per chunk
  static constexpr int kLW = (kIW + kSkWaves - 1) / kSkWaves, kLX = (kIX + kSkWaves - 1) / kSkWaves;  // per wave
  static constexpr int kWB = kIW * 64 * kUW, kXB = kIX * 1024, kStage = kWB + kXB;  // bytes
  // Stages: as many as the budget holds, the 6-bit vmcnt field counts
  // ((S - 1) chunks of loads in flight), and at most six.
  static constexpr int kSL = BUD * 1024 / kStage, kSV = 63 / (kLW + kLX) + 1;
  static constexpr int kS = std::min(std::min(kSL, kSV), 6);
  static constexpr bool kOk = kS >= 2;
  static constexpr int kRing = kOk ? kS * kStage : 1;
  // The waves' sums are added RM activation tiles at a time, in the ring's memory.
  static constexpr int kRedTile = kSkWaves * T * 1024;
  static constexpr int kRM = kRing >= MT * kRedTile                      ? MT
                             : (MT % 4 == 0 && kRing >= 4 * kRedTile)    ? 4
                             : (MT % 2 == 0 && kRing >= 2 * kRedTile)    ? 2
                                                                         : 1;
  static constexpr int kDump = std::max(kRing, kRM * kRedTile);  // 1 KB that surplus loads write
  static constexpr int kLds = kDump + 1024;
};

// Up to kSkGroupMax linears over the same activations in one launch: job j
// owns workgroups begin[j] .. begin[j+1]-1: its row tiles, each split over
// kg[j] consecutive workgroups along K, with arrival counters ctr[j] ..; a
// workgroup's partial tile sits at its own index in the workspace.
constexpr int kSkGroupMax = nfhip::kGemvGroupMax;
static_assert(kSkGroupMax == 4, "skinny_kernel passes begin[1..3] as scalar arguments");
struct SkGroup {
  const uint8_t* W[kSkGroupMax];
  void* C[kSkGroupMax];
  int N[kSkGroupMax];
  int begin[kSkGroupMax + 1];
  int kg[kSkGroupMax];
  int ctr[kSkGroupMax];
};

// Job 0's fields and the job boundaries begin[1..3] come first as plain
// scalars (W0 = grp.W[0], ...), so they are among the arguments preloaded
// into SGPRs at wave launch and a workgroup of job 0 (every workgroup of a
// single launch) starts without a scalar load from the argument block.
template <class QF, typename XT, int MT, int T, int GN, int BUD>
__global__ __launch_bounds__(64 * kSkWaves) void skinny_kernel(const XT* __restrict__ A,
                                                               const uint8_t* __restrict__ W0, int N0, int KG0, int b1,
                                                               int b2, int b3, int M, int K, void* C0, int CTR0,
                                                               float* __restrict__ ws_part,
                                                               uint32_t* __restrict__ ws_cnt, const SkGroup grp) {
  typedef SkGeom<QF, XT, MT, T, GN, BUD> G;
  constexpr bool kF32 = sizeof(XT) == 4;
  constexpr bool kQ4 = SkBlk<QF>::kSlot == 4;
  constexpr int S = G::kS, NT = 64 * kSkWaves;
  const int bx = (int)blockIdx.x;
  const int job = (bx >= b1) + (bx >= b2) + (bx >= b3);
  const uint8_t* __restrict__ W = W0;
  void* Cv = C0;
  int N = N0, wg0 = 0, KG = KG0, ctr0 = CTR0;
  if (job > 0) {
    W = grp.W[job];
    Cv = grp.C[job];
    N = grp.N[job];
    wg0 = grp.begin[job];
    KG = grp.kg[job];
    ctr0 = grp.ctr[job];
  }
  XT* __restrict__ C = static_cast<XT*>(Cv);
  const int local = bx - wg0, tile = local / KG, kg = local - tile * KG;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* const dump = smem + G::kDump;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int gk = wave / GN, gn = wave % GN;
  const int r16 = lane & 15, s = lane >> 4;
  const int NC = (K + G::kCK - 1) / G::kCK;
  const int n0 = tile * G::kBN;
  const int c_begin = (int)((long)NC * kg / KG), c_end = (int)((long)NC * (kg + 1) / KG);
  const uint32_t row_bytes = (uint32_t)(K / 32) * SkBlk<QF>::kBytes;

  // Lane load u of a weight chunk: row u / kUR, unit u % kUR, so consecutive
  // lanes read consecutive bytes of a row; it lands at LDS unit u (rows kRB
  // bytes apart).  Rows past N reload row N-1 (their outputs are never stored).
  uint32_t woff[G::kLW], xoff[G::kLX], wpart[G::kLW], xpart[G::kLX];  // part: byte within the row's chunk
#pragma unroll
  for (int j = 0; j < G::kLW; ++j) {
    const int u = (wave + kSkWaves * j) * 64 + lane;
    int row = u / G::kUR;
    const int part = u - row * G::kUR;
    row = row < G::kBN ? row : G::kBN - 1;
    const int n = n0 + row < N ? n0 + row : N - 1;
    wpart[j] = (uint32_t)(part * G::kUW);
    woff[j] = (uint32_t)n * row_bytes + wpart[j];
  }
  // Lane load u of an activation chunk: row u / kXR, slot u % kXR, which
  // holds the row's 16-byte unit slot ^ (row & 15), so the 16 rows a read
  // takes the same unit of fall in 16 different bank groups.  Rows past M
  // reload row M-1 (an activation row feeds its own output row only).
#pragma unroll
  for (int j = 0; j < G::kLX; ++j) {
    const int u = (wave + kSkWaves * j) * 64 + lane;
    const int row = u / G::kXR, slot = u % G::kXR;
    const int m = row < M ? row : M - 1;
    xpart[j] = (uint32_t)((slot ^ (row & 15)) * 16);
    xoff[j] = (uint32_t)m * (uint32_t)K * (uint32_t)sizeof(XT) + xpart[j];
  }
  const uint32_t w_bytes = (uint32_t)N * row_bytes, x_bytes = (uint32_t)M * (uint32_t)K * (uint32_t)sizeof(XT);
  // Chunk c into stage st.  Every wave issues the same number of loads for
  // every chunk, so the wait counts below are exact: chunks past the range
  // and a wave's surplus loads go through an empty resource (the surplus
  // into the dump), and in a last, partial chunk the units past the row's
  // end are out of range; both read zeros (zero scales and activations).
  auto issue = [&](int c, int st) {
    const bool live = c < c_end;
    const uint32_t wo = (uint32_t)c * (uint32_t)G::kRB, xo = (uint32_t)c * (uint32_t)(G::kCK * sizeof(XT));
    const uint32_t wleft = row_bytes - wo, xleft = (uint32_t)K * (uint32_t)sizeof(XT) - xo;
    uint8_t* const base = smem + st * G::kStage;
#pragma unroll
    for (int j = 0; j < G::kLW; ++j) {
      const int i = wave + kSkWaves * j;
      const bool in = G::kIW % kSkWaves == 0 || i < G::kIW;
      const __amdgpu_buffer_rsrc_t r = sk_rsrc(W, __builtin_amdgcn_readfirstlane(live && in ? w_bytes : 0u));
      sk_dma<G::kUW>(r, in ? base + i * 64 * G::kUW : dump, wpart[j] < wleft ? woff[j] + wo : 0xFFFFFFF0u);
    }
#pragma unroll
    for (int j = 0; j < G::kLX; ++j) {
      const int i = wave + kSkWaves * j;
      const bool in = G::kIX % kSkWaves == 0 || i < G::kIX;
      const __amdgpu_buffer_rsrc_t r = sk_rsrc(A, __builtin_amdgcn_readfirstlane(live && in ? x_bytes : 0u));
      sk_dma<16>(r, in ? base + G::kWB + i * 1024 : dump, xpart[j] < xleft ? xoff[j] + xo : 0xFFFFFFF0u);
    }
  };

  float4v acc[MT][T];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t) acc[mt][t] = float4v{0.f, 0.f, 0.f, 0.f};

  // Operands of one unit of K (a block; a pair of blocks for f16 Q4_0).
  constexpr bool kPair = G::kUB == 2;
  constexpr int QW = (kF32 && kQ4) ? 2 : 3;            // code dwords
  constexpr int XW = (kF32 || kPair) ? 2 : 1;          // 16-byte activation pieces
  struct Ops {
    uint32_t w[T][QW];
    uint16_t d[T];
    u32x4 x[MT][XW];
  };
  auto read_ops = [&](int st, Ops& o) {
    const uint8_t* const xs = smem + st * G::kStage + G::kWB + r16 * (G::kXR * 16);
    // first byte of the lane's block in its row's chunk, and of its codes, less the 2-byte misalignment
    const int bo = kPair ? gk * 36 + 18 * (s >> 1) : gk * SkBlk<QF>::kBytes;
    const int co = kPair ? bo + ((s >> 1) ? 2 : 0) + 8 * (s & 1) : bo + ((gk & 1) ? 2 : 0) + SkBlk<QF>::kSlot * s;
    const uint8_t* const wr = smem + st * G::kStage + (gn * 16 * T + r16) * G::kRB;
    // element offsets of the lane's activations: two pieces of 8 (pair), of 4 (f32), or one of 8
    const int e0 = kPair ? gk * 64 + 32 * (s >> 1) + 8 * (s & 1) : gk * 32 + (kQ4 ? 4 : 8) * s;
    const int e1 = kPair || kQ4 ? e0 + 16 : e0 + 4;
    constexpr int EU = 16 / (int)sizeof(XT);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint8_t* xr = xs + 16 * mt * (G::kXR * 16);
      o.x[mt][0] = *reinterpret_cast<const u32x4*>(xr + ((e0 / EU) ^ r16) * 16);
      if constexpr (XW == 2) o.x[mt][1] = *reinterpret_cast<const u32x4*>(xr + ((e1 / EU) ^ r16) * 16);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const uint32_t* const wc = reinterpret_cast<const uint32_t*>(wr + 16 * t * G::kRB + co);
#pragma unroll
      for (int i = 0; i < QW; ++i) o.w[t][i] = wc[i];
      o.d[t] = *reinterpret_cast<const uint16_t*>(wr + 16 * t * G::kRB + bo);
    }
  };
  auto compute = [&](const Ops& o) {
    // bytes the codes sit into their first dword
    const uint32_t sh = kPair ? ((s >> 1) ? 0u : 2u) : ((gk & 1) ? 0u : 2u);
    if constexpr (kF32) {
      bf16x8 a1[MT], a2[MT];
      float4v b0[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const float4v lo = __builtin_bit_cast(float4v, o.x[mt][0]), hi = __builtin_bit_cast(float4v, o.x[mt][XW - 1]);
        const float xv[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        split2(xv, a1[mt], a2[mt]);
        b0[mt] = float4v{0.f, 0.f, 0.f, 0.f};
        if constexpr (kQ4) {
          const __bf16 c8 = (__bf16)(-136.0f);
          const bf16x8 bc = {c8, c8, c8, c8, c8, c8, c8, c8};
          b0[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[mt], bc, b0[mt], 0, 0, 0);
          b0[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[mt], bc, b0[mt], 0, 0, 0);
        }
      }
#pragma unroll
      for (int t = 0; t < T; ++t) {
        uint32_t q[SkBlk<QF>::kSlot / 4];
#pragma unroll
        for (int i = 0; i + 1 < QW; ++i) q[i] = __builtin_amdgcn_alignbyte(o.w[t][i + 1], o.w[t][i], sh);
        const float d = h2f_bits(o.d[t]);
        const bf16x8 b = sk_b_codes<QF>(q);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          float4v dd = b0[mt];
          dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[mt], b, dd, 0, 0, 0);
          dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[mt], b, dd, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[mt][t][i] = __builtin_fmaf(d, dd[i], acc[mt][t][i]);
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const uint32_t db = o.d[t];
        const half2v d2 = sk_h2(db | (db << 16));
        const uint32_t qa = __builtin_amdgcn_alignbyte(o.w[t][1], o.w[t][0], sh);
        const uint32_t qb = __builtin_amdgcn_alignbyte(o.w[t][QW - 1], o.w[t][1], sh);
        const half8 b0 = sk_b_f16<QF, false>(qa, qb, d2);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, o.x[mt][0]), b0, acc[mt][t], 0, 0, 0);
        if constexpr (kPair) {
          const half8 b1 = sk_b_f16<QF, true>(qa, qb, d2);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, o.x[mt][XW - 1]), b1, acc[mt][t], 0, 0, 0);
        }
      }
    }
  };
  // Iteration i: wait for chunk i (the S-2 younger ones may stay in flight),
  // barrier (every wave's loads of chunk i are in, and every wave is done with
  // chunk i-1, whose stage takes chunk i+S-1), read the wave's operands,
  // issue chunk i+S-1, compute.
  const int nch = c_end - c_begin;
#pragma unroll
  for (int i = 0; i < S - 1; ++i) issue(c_begin + i, i);
  int st = 0;
  for (int i = 0; i < nch; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(sk_wait_imm((S - 2) * (G::kLW + G::kLX)));
    sk_barrier();
    Ops o;
    read_ops(st, o);
    __builtin_amdgcn_sched_barrier(0);
    issue(c_begin + i + S - 1, st == 0 ? S - 1 : st - 1);
    __builtin_amdgcn_sched_barrier(0);
    // One unit a chunk.  As the body of a loop of one pass it is unrolled late,
    // and the compiler orders the unpacking and the activation splits better:
    // f32 Q8_0 M = 17 14336x4096 28.4 -> 26.5 us, f16 Q4_0 M = 32 50257x768
    // 12.4 -> 11.6.
#pragma unroll
    for (int unit = 0; unit < 1; ++unit) {
      __builtin_amdgcn_sched_barrier(0);
      compute(o);
      __builtin_amdgcn_sched_barrier(0);
    }
    st = st + 1 == S ? 0 : st + 1;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  sk_barrier();

  // Add the kGK waves' sums in wave order, RM activation tiles a round; value
  // v of a round is float4 (mt, t, lane) of wave group g.
  constexpr int RM = G::kRM, RQ = GN * RM * T * 64;  // float4 sums per round
  constexpr int VPT = (RQ + NT - 1) / NT;
  constexpr int NQ = GN * MT * T * 64;               // float4 per workgroup tile
  float4v sum[MT / RM][VPT];
#pragma unroll
  for (int rd = 0; rd < MT / RM; ++rd) {
    float4v* const red = reinterpret_cast<float4v*>(smem);
#pragma unroll
    for (int mt = 0; mt < RM; ++mt)
#pragma unroll
      for (int t = 0; t < T; ++t) red[((wave * RM + mt) * T + t) * 64 + lane] = acc[rd * RM + mt][t];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int v = tid + NT * j;
      if (RQ % NT == 0 || v < RQ) {
        const int g = v / (RM * T * 64), w = v - g * (RM * T * 64);
        float4v x = red[g * (RM * T * 64) + w];
#pragma unroll
        for (int k = 1; k < G::kGK; ++k) x += red[(k * GN + g) * (RM * T * 64) + w];
        sum[rd][j] = x;
      }
    }
    if (rd + 1 < MT / RM) __syncthreads();
  }
  auto store = [&](int rd, int j, float4v x) {
    const int v = tid + NT * j;
    const int l = v & 63, t = (v >> 6) % T, mt = (v >> 6) / T % RM + rd * RM, g = v / (RM * T * 64);
    const int n = n0 + (g * T + t) * 16 + (l & 15), m = 16 * mt + 4 * (l >> 4);
    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (m + i < M) C[(size_t)(m + i) * N + n] = (XT)x[i];
  };
  if (KG > 1) {
    // K split across workgroups: park this tile (sc1 stores), count arrivals;
    // the last workgroup adds the KG tiles in order kg = 0..KG-1, the loads of
    // up to GB tiles in flight together, and resets the counter.
    const CoherentTile tws(reinterpret_cast<float4v*>(ws_part) + (size_t)(wg0 + tile * KG) * NQ, (uint32_t)(KG * NQ * 16));
#pragma unroll
    for (int rd = 0; rd < MT / RM; ++rd)
#pragma unroll
      for (int j = 0; j < VPT; ++j)
        if (RQ % NT == 0 || tid + NT * j < RQ) tws.store((uint32_t)(kg * NQ + rd * RQ + j * NT + tid), sum[rd][j]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    __shared__ uint32_t is_last;
    if (tid == 0) {
      const uint32_t prev = __hip_atomic_fetch_add(&ws_cnt[ctr0 + tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      is_last = prev == (uint32_t)(KG - 1);
    }
    __syncthreads();
    if (!is_last) return;
    constexpr int VT = VPT * (MT / RM);
    constexpr int GB = VT >= 16 ? 1 : 16 / VT;
    for (int g0 = 0; g0 < KG; g0 += GB) {
      float4v p[GB][MT / RM][VPT];
#pragma unroll
      for (int gb = 0; gb < GB; ++gb)
        if (g0 + gb < KG) {
#pragma unroll
          for (int rd = 0; rd < MT / RM; ++rd)
#pragma unroll
            for (int j = 0; j < VPT; ++j) p[gb][rd][j] = tws.load((uint32_t)((g0 + gb) * NQ + rd * RQ + j * NT + (RQ % NT == 0 || tid + NT * j < RQ ? tid : 0)));
        }
#pragma unroll
      for (int gb = 0; gb < GB; ++gb)
        if (g0 + gb < KG) {
#pragma unroll
          for (int rd = 0; rd < MT / RM; ++rd)
#pragma unroll
            for (int j = 0; j < VPT; ++j) sum[rd][j] = g0 + gb == 0 ? p[gb][rd][j] : sum[rd][j] + p[gb][rd][j];
        }
    }
    if (tid == 0) __hip_atomic_store(&ws_cnt[ctr0 + tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int rd = 0; rd < MT / RM; ++rd)
#pragma unroll
    for (int j = 0; j < VPT; ++j)
      if (RQ % NT == 0 || tid + NT * j < RQ) store(rd, j, sum[rd][j]);
}

// ---- host ------------------------------------------------------------------

// Launch time in microseconds (relative use only): the chunks a workgroup
// runs one after the other, each as long as its CU's workgroups compute (a
// constant, 1024s of codes, KB of activations, 1024s of code x 16-row tile
// products) or as the loads in flight take to arrive; further rounds of
// workgroups; the fix-up of a K split; no less than the bytes at the rate
// the stream reaches.  The coefficients are least-squares fits to about 700
// launches per format and type on MI355X (16 shapes from 512 x 1024 to 28672
// x 8192, 4 to 128 rows, every variant, 1 to 8 K splits).  Over the 35 shapes
// of profiles/skinny_variant_sweep.csv the pick is within 0.2-8 % of the
// fastest on average (worst 1.30 x: f16 Q8_0 2048x2048 M = 32).
struct SkCost {
  float chunk, codes, xkb, prod;  // per chunk
  float base, split, round, tbs;  // launch, K split, further rounds; TB/s
  float red, part, lat;           // wave sums (KB), partial tiles (MB), load latency
};
template <class QF, typename XT> struct SkCostOf;
template <> struct SkCostOf<Q4_0, half_t> {
  static constexpr SkCost k = {0.0362f, 0.0229f, 0.0105f, 0.0038f, 2.14f, 0.81f, 2.55f, 3.93f, 0.0096f, 0.576f, 1.4f};
};
template <> struct SkCostOf<Q8_0, half_t> {
  static constexpr SkCost k = {0.146f, 0.0326f, 0.0034f, 0.0072f, 2.43f, 0.89f, 2.57f, 21.f, 0.0023f, 0.563f, 1.4f};
};
template <> struct SkCostOf<Q4_0, float> {
  static constexpr SkCost k = {0.148f, 0.0013f, 0.0065f, 0.0221f, 1.77f, 0.93f, 2.51f, 3.11f, 0.0076f, 0.661f, 1.4f};
};
template <> struct SkCostOf<Q8_0, float> {
  static constexpr SkCost k = {0.0488f, 0.0204f, 0.0114f, 0.02f, 1.0f, 1.06f, 2.36f, 4.5f, 0.0083f, 0.7f, 1.4f};
};

// Jobs of one launch: rows and K splits (kg[j] = 0: none chosen yet).
struct SkJobs {
  uint32_t n = 0;
  uint32_t N[kSkGroupMax];
  int kg[kSkGroupMax];
};

template <class QF, typename XT, int MT, int T, int GN, int BUD>
float sk_cost(const SkJobs& jobs, uint32_t K) {
  typedef SkGeom<QF, XT, MT, T, GN, BUD> G;
  constexpr SkCost c = SkCostOf<QF, XT>::k;
  constexpr long per_cu = BUD > 79 ? 1 : BUD > 53 ? 2 : 3, kCUs = 256;
  const int NC = (int)((K + G::kCK - 1) / G::kCK);
  long wgs = 0, split_wgs = 0, rows = 0;
  int chunks = 0, kg = 1;
  for (uint32_t j = 0; j < jobs.n; ++j) {
    const long w = ((long)jobs.N[j] + G::kBN - 1) / G::kBN * jobs.kg[j];
    wgs += w;
    rows += jobs.N[j];
    if (jobs.kg[j] > 1) split_wgs += w;
    chunks = std::max(chunks, (NC + jobs.kg[j] - 1) / jobs.kg[j]);
    kg = std::max(kg, jobs.kg[j]);
  }
  const long rounds = (wgs + per_cu * kCUs - 1) / (per_cu * kCUs), on_cu = std::min((wgs + kCUs - 1) / kCUs, per_cu);
  constexpr float codes = G::kBN * G::kCK / 1024.f;
  const float tc = c.chunk + c.codes * codes + c.xkb * (G::kXB / 1024.f) + c.prod * MT * codes;
  float t = c.base + (float)(rounds * chunks) * std::max(tc * (float)on_cu, c.lat / (G::kS - 1)) +
            c.round * (float)(rounds - 1) + c.red * (kSkWaves * T * MT);
  int l2 = 0;
  while ((2 << l2) <= kg) ++l2;
  if (kg > 1) t += c.split * (float)(1 + l2) + c.part * (float)split_wgs * (MT * 16 * G::kBN * 4) * 1e-6f;
  const float bytes = c.base + (float)rows * (float)(K / 32) * SkBlk<QF>::kBytes / (c.tbs * 1e6f);
  return std::max(t, bytes) + 0.02f * t;
}

// A launch's variant (index into sk_variants' list for its MT), the order of
// its sums (GN) and its K split.
struct SkPick {
  float key = 1e30f;
  int variant = -1, order = 0, kg = 1;
};

template <class QF, typename XT, int MT, int T, int GN, int BUD>
void sk_try(int index, uint32_t N, uint32_t K, const nfhip::Workspace& ws, SkPick& best) {
  typedef SkGeom<QF, XT, MT, T, GN, BUD> G;
  if constexpr (G::kOk) {
    const long tiles = ((long)N + G::kBN - 1) / G::kBN;
    const int NC = (int)((K + G::kCK - 1) / G::kCK);
    // A split that gains a launch of its own little costs the launch it
    // shares with larger jobs more: Q8_0 f32 M = 8, q (4096), k and v (1024
    // rows) at K = 4096 15.7 us without this margin, 12.6 with it.
    constexpr float less = MT <= 2 ? 0.06f : 0.f;
    for (int kg = 1, l2 = 0; kg <= 8 && kg <= NC; kg *= 2, ++l2) {
      if (kg > 1 && (tiles > (long)ws.cnt_len || (size_t)tiles * kg * (MT * 16 * G::kBN) > ws.part_floats)) break;
      const float t = sk_cost<QF, XT, MT, T, GN, BUD>(SkJobs{1, {N}, {kg}}, K);
      const float key = t * (1.f + less * l2);
      if (key < best.key) best = SkPick{key, index, GN, kg};
    }
  }
}

// One launch for n jobs (n = 1: a single linear) with variant <T, GN, BUD> and
// each job's own K split.
template <class QF, typename XT, int MT, int T, int GN, int BUD>
hipError_t sk_launch(const XT* A, const nfhip::GemvJob* jobs, const int* kg, uint32_t n, uint32_t M, uint32_t K,
                     const nfhip::Workspace& ws, hipStream_t s) {
  typedef SkGeom<QF, XT, MT, T, GN, BUD> G;
  if constexpr (!G::kOk) {
    return hipErrorNotSupported;
  } else {
    SkGroup grp{};
    long wgs = 0, tiles = 0;
    bool split = false;
    for (uint32_t j = 0; j < n; ++j) {
      const long t = ((long)jobs[j].N + G::kBN - 1) / G::kBN;
      split = split || kg[j] > 1;
      grp.W[j] = static_cast<const uint8_t*>(jobs[j].W);
      grp.C[j] = jobs[j].C;
      grp.N[j] = (int)jobs[j].N;
      grp.begin[j] = (int)wgs;
      grp.kg[j] = kg[j];
      grp.ctr[j] = (int)tiles;
      wgs += t * kg[j];
      tiles += t;
    }
    if (split && (tiles > (long)ws.cnt_len || (size_t)wgs * (MT * 16 * G::kBN) > ws.part_floats))
      return hipErrorNotSupported;
    for (int q = (int)n; q <= kSkGroupMax; ++q) grp.begin[q] = (int)wgs;
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&skinny_kernel<QF, XT, MT, T, GN, BUD>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, G::kLds);
    if (attr != hipSuccess) return attr;
    skinny_kernel<QF, XT, MT, T, GN, BUD><<<dim3((unsigned)wgs), dim3(64 * kSkWaves), G::kLds, s>>>(
        A, grp.W[0], grp.N[0], grp.kg[0], grp.begin[1], grp.begin[2], grp.begin[3], (int)M, (int)K, grp.C[0],
        grp.ctr[0], ws.part, ws.cnt, grp);
    return hipGetLastError();
  }
}

// Whether a variant is for rows of this K.  The 52 KB rings (two stages, three
// workgroups per CU) are for weight rows of at most 768 bytes: such a row is
// one to a few chunks, a deeper ring is never full, and what bounds a matrix
// of many of them is the number of workgroups loading at once.  us at M = 8
// with 78 KB rings -> with these: Q4_0 f32 128256x256 16.2 -> 12.0, 50257x768
// 14.8 -> 13.2, f16 50257x768 12.9 -> 10.1, 128256x768 30.0 -> 24.8, Q8_0 f16
// 65536x512 14.4 -> 12.9; past that the deeper rings win: Q8_0 f16 50257x1024
// 18.2 against 19.6, f32 50257x768 16.3 against 17.1.
template <class QF, int BUD>
bool sk_suits(uint32_t K) {
  return BUD > 53 || K / 32 * SkBlk<QF>::kBytes <= 768;
}

// The variants of each MT: f(index, T, GN, BUD), integral constants.
// One activation tile: two or three workgroups per CU; four and eight: one,
// and more waves along N, so that each activation operand read from LDS feeds
// more weight tiles.
template <int MT, class F>
void sk_variants(F&& f) {
#define SK_V(i, t, gn, bud)                                                                                \
  f(std::integral_constant<int, i>{}, std::integral_constant<int, t>{}, std::integral_constant<int, gn>{}, \
    std::integral_constant<int, bud>{})
  if constexpr (MT == 1) {
    SK_V(0, 1, 1, 78);
    SK_V(1, 2, 1, 78);
    SK_V(2, 4, 1, 78);
    SK_V(3, 2, 2, 78);
    SK_V(4, 4, 1, 52);
    SK_V(5, 4, 2, 52);
  } else if constexpr (MT == 2) {
    SK_V(0, 1, 1, 78);
    SK_V(1, 2, 1, 78);
    SK_V(2, 2, 1, 158);
    SK_V(3, 4, 1, 158);
    SK_V(4, 2, 2, 78);
    SK_V(5, 4, 2, 78);
    SK_V(6, 4, 2, 52);
  } else {
    SK_V(0, 1, 1, 158);
    SK_V(1, 2, 1, 158);
    SK_V(2, 4, 1, 158);
    SK_V(3, 2, 2, 158);
    SK_V(4, 4, 2, 158);
  }
#undef SK_V
}

template <class QF, typename XT, int MT>
SkPick sk_pick(uint32_t N, uint32_t K, const nfhip::Workspace& ws) {
  SkPick best;
  sk_variants<MT>([&](auto i, auto t, auto gn, auto bud) {
    // f32: one order of sums for all but the tallest weights, so the linears
    // of a layer share a launch (Q8_0 M = 8, q, k and v of 4096, 1024 and
    // 1024 rows: 20.9 us when q alone took two waves along N); at 50257x768
    // M = 32 the two waves along N take 27.3 -> 19.2 us (Q4_0).
    const bool order_ok = sizeof(XT) == 2 || gn() == (N > 16384 ? 2 : 1) || (N > 16384 && MT == 1);
    if (order_ok && sk_suits<QF, bud()>(K)) sk_try<QF, XT, MT, t(), gn(), bud()>(i(), N, K, ws, best);
  });
  return best;
}

// A group of jobs: each with the K split of its own pick, all with the
// variant the cost model finds fastest for the whole among those of the
// picks' order.  An output depends on GN and the K split (the order of
// its sums) but not on T or the ring's depth, so a job gets the bits of its
// own launch.  Declined (hipErrorNotSupported: the caller splits the group)
// only when the picks differ in order or the partial tiles do not fit: K
// splits chosen for single launches can add up to further rounds of
// workgroups, but one launch measured faster than one each all the same, us
// apart / together: f32 M = 17, q, k and v of 8192, 1024 and 1024 rows at K =
// 8192 Q4_0 36.7 / 34.8, Q8_0 41.4 / 39.0, two 14336x4096 44.5 / 43.0 and
// 53.0 / 51.4; f16 M = 16, two 28672x8192 72.1 / 69.1 and 111.9 / 105.5; the
// exception found, Q8_0 f16 M = 17, that q, k and v: 34.5 / 37.4.
template <class QF, typename XT, int MT>
hipError_t sk_group(const XT* A, const nfhip::GemvJob* jobs, uint32_t n, uint32_t M, uint32_t K,
                    const nfhip::Workspace& ws, hipStream_t s) {
  SkJobs js;
  js.n = n;
  SkPick pick;
  for (uint32_t j = 0; j < n; ++j) {
    const SkPick p = sk_pick<QF, XT, MT>(jobs[j].N, K, ws);
    if (p.variant < 0 || (j > 0 && p.order != pick.order)) return hipErrorNotSupported;
    js.N[j] = jobs[j].N;
    js.kg[j] = p.kg;
    pick = p;
  }
  if (n > 1) {
    float best = 1e30f;
    sk_variants<MT>([&](auto i, auto t, auto gn, auto bud) {
      if constexpr (SkGeom<QF, XT, MT, t(), gn(), bud()>::kOk) {
        const float c = sk_cost<QF, XT, MT, t(), gn(), bud()>(js, K);
        if (gn() == pick.order && sk_suits<QF, bud()>(K) && c < best) best = c, pick.variant = i();
      }
    });
  }
  hipError_t e = hipErrorNotSupported;
  sk_variants<MT>([&](auto i, auto t, auto gn, auto bud) {
    if (i() == pick.variant) e = sk_launch<QF, XT, MT, t(), gn(), bud()>(A, jobs, js.kg, n, M, K, ws, s);
  });
  return e;
}

template <class QF, typename XT>
hipError_t sk_dispatch(const void* A, const nfhip::GemvJob* jobs, uint32_t n, uint32_t M, uint32_t K,
                       const nfhip::Workspace& ws, hipStream_t s) {
  const XT* a = static_cast<const XT*>(A);
  if (M <= 16) return sk_group<QF, XT, 1>(a, jobs, n, M, K, ws, s);
  if (M <= 32) return sk_group<QF, XT, 2>(a, jobs, n, M, K, ws, s);
  if (M <= 64) return sk_group<QF, XT, 4>(a, jobs, n, M, K, ws, s);
  if constexpr (sizeof(XT) == 2) return sk_group<QF, XT, 8>(a, jobs, n, M, K, ws, s);
  return hipErrorNotSupported;
}

}  // namespace nfk

namespace nfhip {

hipError_t launch_skinny_group(QFmt q, EType t, const void* A, const GemvJob* jobs, uint32_t n, uint32_t M,
                               uint32_t K, const Workspace& ws, hipStream_t s) {
  if (M > skinny_max_rows(t) || n < 1 || n > (uint32_t)kGemvGroupMax) return hipErrorNotSupported;
  const bool ring = ring_serves(q, t, M, jobs[0].N, K);
  for (uint32_t j = 0; j < n; ++j)
    if (!skinny_fits(M, jobs[j].N, K, A, jobs[j].W) || ring_serves(q, t, M, jobs[j].N, K) != ring)
      return hipErrorNotSupported;
  if (ring) return launch_skinny_ring(q, A, jobs, n, M, K, ws, s);
  if (q == QFmt::Q4_0)
    return t == EType::F32 ? nfk::sk_dispatch<nfk::Q4_0, float>(A, jobs, n, M, K, ws, s)
                           : nfk::sk_dispatch<nfk::Q4_0, nfk::half_t>(A, jobs, n, M, K, ws, s);
  return t == EType::F32 ? nfk::sk_dispatch<nfk::Q8_0, float>(A, jobs, n, M, K, ws, s)
                         : nfk::sk_dispatch<nfk::Q8_0, nfk::half_t>(A, jobs, n, M, K, ws, s);
}

bool skinny_fits(uint32_t M, uint32_t N, uint32_t K, const void* A, const void* W) {
  // 32-bit in-kernel offsets: weight matrix and activation tile below 4 GB;
  // K % 256 == 0 keeps rows and their chunks on 16-byte boundaries
  const uint64_t wbytes = (uint64_t)N * (K / 32) * 34, abytes = (uint64_t)128 * K * 4;
  return M >= 1 && M <= 128 && K % 256 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 &&
         wbytes < 0xFFFFFFF0ull && abytes < 0xFFFFFFF0ull;
}

// Activation rows per launch: four 16-row tiles of f32 (two bf16 pieces
// each), eight of f16.
uint32_t skinny_max_rows(EType t) { return t == EType::F32 ? 64u : 128u; }

hipError_t launch_skinny(QFmt q, EType t, const void* A, const void* W, void* C, uint32_t M, uint32_t N,
                         uint32_t K, const Workspace& ws, hipStream_t s) {
  const GemvJob job{W, C, N};
  return launch_skinny_group(q, t, A, &job, 1, M, K, ws, s);
}

}  // namespace nfhip
