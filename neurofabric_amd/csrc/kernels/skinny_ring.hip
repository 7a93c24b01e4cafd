// skinny_ring.hip — fused dequant + matmul of up to 64 f32 activation rows on
// MFMA, weights streamed through an LDS ring (33 rows and more, mostly).
//
// The same products as skinny.hip's f32 path (activations split into two
// bf16 parts, exact bf16 codes, the block scale applied per block in fp32),
// split for weights with many rows: every wave of a workgroup owns weight
// rows and walks the workgroup's whole K range, in chunks of 64 elements, so
// the workgroup needs 32 KB of split activations and a small weight ring and
// two fit on a CU (with one or two 16-row tiles a wave; from 65536 rows on,
// with four, one); skinny.hip's workgroups for these batches (whole
// 256-element activation chunks in the ring) fill one.  Bound by the fp32
// scale FMAs and unpacking beside the MFMAs.  ring_serves() has the line
// between the two, with both sides' times.
//
// MFMA v_mfma_f32_16x16x32 (bf16): A = activations (16 rows of M), B =
// weights (16 rows of N), D[m][n] = sum over 32 k.  Lane l:
//   A: row l%16, eight k values of slot s = l/16;
//   B: weight row l%16, the same eight k values;
//   D: weight row l%16, activation rows 4s..4s+3.
// Slot s holds the k values a lane unpacks from one code word: Q4_0
// qs[4s..4s+3], i.e. k = 4s..4s+3 (low nibbles) and 16+4s..16+4s+3 (high
// nibbles); Q8_0 codes 8s..8s+7.
#include <algorithm>

#include "../launch.hpp"
#include "common.hpp"

namespace nfk {
namespace ring {

template <class QF> struct SkW;
template <> struct SkW<Q4_0> {
  static constexpr int kPairBytes = 36, kLoads = 5;
};
template <> struct SkW<Q8_0> {
  static constexpr int kPairBytes = 68, kLoads = 7;
};

template <class QF>
__device__ __forceinline__ uint32_t sk_scale_bits(const uint32_t (&w)[SkW<QF>::kLoads], int h) {
  if constexpr (SkW<QF>::kLoads == 5) return h == 0 ? (w[3] & 0xFFFFu) : (w[4] >> 16);
  else return h == 0 ? (w[5] & 0xFFFFu) : (w[6] >> 16);
}

// B operand, f32 path: the codes of the lane's slot as exact bf16 (Q4_0:
// 128 + n with n the unsigned nibble, bf16 0x43nn; Q8_0: the signed code).
template <class QF>
__device__ __forceinline__ bf16x8 sk_b_codes(const uint32_t (&w)[SkW<QF>::kLoads], int h) {
  u32x4 o;
  if constexpr (SkW<QF>::kLoads == 5) {
    const uint32_t q = h == 0 ? __builtin_amdgcn_alignbyte(w[1], w[0], 2) : w[2];
    const uint32_t l = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
    o.x = __builtin_amdgcn_perm(0x43434343u, l, 0x04010400u);   // k = 4s, 4s+1
    o.y = __builtin_amdgcn_perm(0x43434343u, l, 0x04030402u);   // 4s+2, 4s+3
    o.z = __builtin_amdgcn_perm(0x43434343u, hi, 0x04010400u);  // 16+4s, 16+4s+1
    o.w = __builtin_amdgcn_perm(0x43434343u, hi, 0x04030402u);  // 16+4s+2, 16+4s+3
  } else {
    const uint32_t qa = h == 0 ? __builtin_amdgcn_alignbyte(w[1], w[0], 2) : w[3];
    const uint32_t qb = h == 0 ? __builtin_amdgcn_alignbyte(w[2], w[1], 2) : w[4];
    o.x = pack_hi16((float)(int8_t)qa, (float)(int8_t)(qa >> 8));
    o.y = pack_hi16((float)(int8_t)(qa >> 16), (float)((int32_t)qa >> 24));
    o.z = pack_hi16((float)(int8_t)qb, (float)(int8_t)(qb >> 8));
    o.w = pack_hi16((float)(int8_t)(qb >> 16), (float)((int32_t)qb >> 24));
  }
  return __builtin_bit_cast(bf16x8, o);
}

constexpr int kSkGroupMax = nfhip::kGemvGroupMax;
static_assert(kSkGroupMax == 4, "the kernel passes begin[1..3] as scalar arguments");

// Arguments of the kernel: job 0's fields and the job
// boundaries begin[1..3] come first as plain scalars (W0 = grp.W[0], ...),
// so they are among the arguments preloaded into SGPRs at wave launch and a
// workgroup of job 0 (every workgroup of a single launch) issues its first
// loads without a scalar load from the argument block; other jobs read
// their entries of `grp`.  begin[] is non-decreasing and its unused entries
// equal the number of workgroups (tiles) along x.
__device__ __forceinline__ int group_job(int b1, int b2, int b3) {
  const int bx = (int)blockIdx.x;
  return (bx >= b1) + (bx >= b2) + (bx >= b3);
}

// A workgroup is 8 waves (two per SIMD) over 128*T weight rows (wave w: rows
// 16T*w .. 16T*w + 16T-1 as T 16-row tiles), and all waves walk the same K
// range chunk by chunk; a chunk is a pair of blocks (64 elements).  The weight
// ring has S stages; chunk i+S-1 is requested while chunk i is computed, by
// buffer_load ... lds, which writes LDS without passing through registers
// (so S-1 chunks in flight cost no registers), range-checked: chunks past
// the workgroup's range read through a resource of zero bytes (zeros, no
// memory traffic).  A weight row's staged pairs are 9 (17) dwords apart, an
// odd stride, so the 16 rows of a tile read 16 different banks.
//
// The activations (16*MT rows, rows past M repeating row M-1, whose outputs
// are never stored) are L2-resident: each thread loads the 8 values of its
// A operand(s) of chunk i+1 into registers while chunk i computes, and after
// chunk i splits them once for the whole workgroup into the two bf16 pieces
// of the MFMA operand (x ~ b1 + b2, split2), stored in operand order in one
// of two LDS buffers, so a wave reads each piece with one conflict-free
// ds_read_b128.  Every wave then runs the MFMA chain on its tiles (exact bf16
// codes, two chained MFMAs, the block scale applied per block in fp32).
//
// With K split over KG workgroups, each parks its partial tile and
// the last to arrive adds the KG tiles in order kg = 0..KG-1 (deterministic)
// and stores C.
template <class QF, int MT, int T>
struct RingGeom {
  static constexpr int kWaves = 8;
  static constexpr int kPB = SkW<QF>::kPairBytes, kPD = kPB / 4;
  static constexpr int kRW = 16 * T;                   // weight rows per wave
  static constexpr int kWRow = kPD;                    // dwords per staged weight row
  static constexpr int kWDw = kRW * kWRow;             // weight dwords of a wave per chunk
  static constexpr int kJW = (kWDw + 63) / 64;         // dword loads per lane per chunk
  // A wave's area in a stage is padded to whole loads: every lane issues all
  // kJW loads (lanes past kWDw reload the last dword into the padding), so
  // no load sits behind a lane-dependent branch, which made the compiler's
  // wait analysis drop count and wait for loads issued an iteration later.
  static constexpr int kWArea = kJW * 64;
  static constexpr int kStage = kWaves * kWArea;       // dwords of a stage
  static constexpr int kUnits = 2 * MT * 64;           // A operands (lane slots) per chunk
  static constexpr int kUPT = (kUnits + 511) / 512;    // A operands per thread
  static constexpr int kXB = kUnits * 8;               // dwords of one split buffer (two bf16x8 each)
};

// Jobs of one ring launch: job j owns workgroups begin[j] .. begin[j+1]-1,
// tiles[j] row tiles with its own K split kg[j] (tile-major: the kg[j]
// workgroups of a tile are consecutive), and arrival counters
// ctr[j] .. ctr[j] + tiles[j] - 1; a workgroup's partial tile sits at its
// own index in the workspace.
struct RingGroup {
  const uint8_t* W[kSkGroupMax];
  void* C[kSkGroupMax];
  int N[kSkGroupMax];
  int begin[kSkGroupMax + 1];
  int kg[kSkGroupMax];
  int ctr[kSkGroupMax];
};

// Partial-tile loads (float4 per thread) the split-K fix-up keeps in flight.
constexpr int kRingGatherF4 = 16;

// Arguments: job 0's fields first (W0 = grp.W[0], N0,
// KG0 = grp.kg[0], C0, CTR0 = grp.ctr[0]).
template <class QF, int MT, int T, int S>
__global__ __launch_bounds__(512) void skinny_ring_kernel(const float* __restrict__ A,
                                                         const uint8_t* __restrict__ W0, int N0, int KG0, int b1,
                                                         int b2, int b3, int M, int K, void* C0, int CTR0,
                                                         float* __restrict__ ws_part,
                                                         uint32_t* __restrict__ ws_cnt, const RingGroup grp) {
  const int job = group_job(b1, b2, b3);
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
  float* __restrict__ C = static_cast<float*>(Cv);
  const int local = (int)blockIdx.x - wg0, tile = local / KG, kg = local - tile * KG;
  typedef RingGeom<QF, MT, T> G;
  constexpr bool kQ4 = SkW<QF>::kLoads == 5;
  constexpr int WL = SkW<QF>::kLoads;
  constexpr int RW = G::kRW, NW = G::kWaves, UPT = G::kUPT;
  static_assert(S >= 3 && (S - 2) * G::kJW <= 63, "ring depth and the vmcnt field");
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  uint32_t* const xb0 = smem + S * G::kStage;  // split operands, two buffers of kXB dwords

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, s = lane >> 4;
  const int NC = K >> 6;
  const int n0 = tile * (NW * RW) + wave * RW;  // this wave's first row
  const int c_begin = (int)((long)NC * kg / KG), c_end = (int)((long)NC * (kg + 1) / KG);

  // Weight loads: dword f = lane + 64j of the wave's RW x kWRow chunk is row
  // f / kWRow, dword f % kWRow (pairs of a row are contiguous, so the byte
  // offset within the row is 4 * (f % kWRow)); it lands at LDS dword f.
  const uint32_t row_bytes = (uint32_t)(K >> 6) * G::kPB;
  uint32_t wsrc[G::kJW];
#pragma unroll
  for (int j = 0; j < G::kJW; ++j) {
    const int f = lane + 64 * j < G::kWDw ? lane + 64 * j : G::kWDw - 1;
    const int row = f / G::kWRow, dw = f % G::kWRow;
    const int n = n0 + row < N ? n0 + row : N - 1;
    wsrc[j] = (uint32_t)n * row_bytes + (uint32_t)(4 * dw);
  }
  const uint32_t w_bytes = (uint32_t)N * row_bytes;
  auto fetch_w = [&](int c, int st) {
    const bool live = c < c_end;
    const __amdgpu_buffer_rsrc_t rw = sk_rsrc(W, __builtin_amdgcn_readfirstlane(live ? w_bytes : 0u));
    const uint32_t wo = __builtin_amdgcn_readfirstlane(live ? (uint32_t)c * (uint32_t)G::kPB : 0u);
    uint32_t* wsb = smem + st * G::kStage + wave * G::kWArea;
#pragma unroll
    for (int j = 0; j < G::kJW; ++j) sk_dma<4>(rw, wsb + 64 * j, wsrc[j], wo);
  };

  // A operands: unit u = (h * MT + mt) * 64 + l is the operand of lane l (row
  // 16mt + l%16, slot l/16) for block h of a chunk: activations k = 32h +
  // {off0 .. off0+3, off1 .. off1+3} of its row (the k order of the lane's
  // weight codes).  Thread tid takes units tid,
  // tid + 512, ...; piece k (0: hi, 1: lo) of unit u goes to 16-byte slot
  // ((u / 64) * 2 + k) * 64 + l of a split buffer, so a wave's read of one
  // piece covers 1 KB contiguously.
  uint32_t xoff[UPT];
  bool xlive[UPT];
#pragma unroll
  for (int k = 0; k < UPT; ++k) {
    const int u = tid + 512 * k;
    xlive[k] = G::kUnits % 512 == 0 || u < G::kUnits;
    const int uu = xlive[k] ? u : 0;
    const int l = uu & 63, mt = (uu >> 6) % MT, h = (uu >> 6) / MT;
    const int m = 16 * mt + (l & 15);
    const int mm = m < M ? m : M - 1;
    xoff[k] = ((uint32_t)mm * (uint32_t)K + (uint32_t)(32 * h + (kQ4 ? 4 : 8) * (l >> 4))) * 4u;
  }
  const uint32_t x_bytes = (uint32_t)M * (uint32_t)K * 4u;
  typedef float4v XSet[UPT][2];
  XSet xr[2];  // activations of two chunks in registers (two chunks ahead)
  auto load_x = [&](int c, XSet& x) {
    const bool live = c < c_end;
    const __amdgpu_buffer_rsrc_t rx = sk_rsrc(A, __builtin_amdgcn_readfirstlane(live ? x_bytes : 0u));
    const uint32_t xo = __builtin_amdgcn_readfirstlane(live ? (uint32_t)c * 256u : 0u);
#pragma unroll
    for (int k = 0; k < UPT; ++k) {
      x[k][0] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(rx, xoff[k], xo, 0));
      x[k][1] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(rx, xoff[k] + (kQ4 ? 64u : 16u), xo, 0));
    }
  };
  auto split_x = [&](uint32_t* xb, const XSet& x) {
#pragma unroll
    for (int k = 0; k < UPT; ++k) {
      if (xlive[k]) {
        const int u = tid + 512 * k;
        const float xv[8] = {x[k][0].x, x[k][0].y, x[k][0].z, x[k][0].w,
                             x[k][1].x, x[k][1].y, x[k][1].z, x[k][1].w};
        bf16x8 a1, a2;
        split2(xv, a1, a2);
        uint32_t* dst = xb + (((u >> 6) * 2) * 64 + (u & 63)) * 4;
        *reinterpret_cast<bf16x8*>(dst) = a1;
        *reinterpret_cast<bf16x8*>(dst + 256) = a2;
      }
    }
  };

  bool wvalid[T];
#pragma unroll
  for (int t = 0; t < T; ++t) wvalid[t] = n0 + 16 * t + r16 < N;

  float4v acc[MT][T];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t) acc[mt][t] = float4v{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int st, const uint32_t* xb) {
    const uint32_t* wsb = smem + st * G::kStage + wave * G::kWArea;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 a1[MT], a2[MT];
      float4v base[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint32_t* up = xb + (((h * MT + mt) * 2) * 64 + lane) * 4;
        a1[mt] = *reinterpret_cast<const bf16x8*>(up);
        a2[mt] = *reinterpret_cast<const bf16x8*>(up + 256);
        base[mt] = float4v{0.f, 0.f, 0.f, 0.f};
        if constexpr (kQ4) {
          // sum_k (-136) * x, the offset of the 128 + n codes, shared by
          // all weight tiles
          const __bf16 c8 = (__bf16)(-136.0f);
          const bf16x8 bc = {c8, c8, c8, c8, c8, c8, c8, c8};
          base[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[mt], bc, base[mt], 0, 0, 0);
          base[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[mt], bc, base[mt], 0, 0, 0);
        }
      }
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const uint32_t* pr = wsb + (16 * t + r16) * G::kWRow;
        uint32_t w[WL];
        if constexpr (WL == 5) {
          w[0] = pr[s];      // block 0 codes, realigned with w[1]
          w[1] = pr[s + 1];
          w[2] = pr[5 + s];  // block 1 codes
          w[3] = pr[0];      // block 0 scale (low half)
          w[4] = pr[4];      // block 1 scale (high half)
        } else {
          w[0] = pr[2 * s];  // block 0 codes: bytes 2+8s .. 9+8s across three dwords
          w[1] = pr[2 * s + 1];
          w[2] = pr[2 * s + 2];
          w[3] = pr[9 + 2 * s];  // block 1 codes
          w[4] = pr[10 + 2 * s];
          w[5] = pr[0];      // block 0 scale (low half)
          w[6] = pr[8];      // block 1 scale (high half)
        }
        const bf16x8 b = sk_b_codes<QF>(w, h);
        float d = h2f_bits((uint16_t)sk_scale_bits<QF>(w, h));
        if (!wvalid[t]) d = 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          float4v dd = base[mt];
          dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[mt], b, dd, 0, 0, 0);
          dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[mt], b, dd, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[mt][t][i] = __builtin_fmaf(d, dd[i], acc[mt][t][i]);
        }
      }
    }
  };

  // Pipeline.  Before the loop: chunk 0's activations, the weights of
  // chunks c_begin .. c_begin+S-3, chunk 1's activations and chunk S-2's
  // weights go out, in that order (the order of the loop's own issue, so the
  // loads pending at the loop entry match those pending around the loop and
  // the compiler's waits stay exact), and chunk 0 is split.  Iteration i
  // (activation register set p = i & 1):
  //   wait for chunk i's weights and for its own split stores, then one
  //   barrier makes chunk i's weights and split operands visible and retires
  //   chunk i-1 (its stage receives chunk i+S-1, its split buffer the split
  //   of chunk i+1);
  //   chunk i+2's activations are requested into set p (chunk i's, split in
  //   iteration i-1), then chunk i+S-1's weights;
  //   chunk i computes, and chunk i+1 (set p^1, requested one iteration
  //   earlier) is split.
  // Loads complete in issue order, so the activations are requested two
  // chunks ahead: the split's wait then covers only loads issued an
  // iteration earlier (with them one chunk ahead, it also waited for the
  // weight loads issued just before them).  Measured on MI355X with the
  // batched fix-up below (same box, against the previous kernel): Llama-3-8B
  // Q8_0 decode step 5.31 -> 5.17 ms at M = 64, 3.32 -> 3.11 ms at M = 16,
  // TinyLlama Q4_0 M = 16 961 -> 940 us; 14336 x 4096 at M = 64 stays at
  // about 1.4 us per chunk, which the load order therefore does not set.  Every thread issues the same loads per
  // chunk (2 * UPT activation, kJW weight), so the counts below are exact:
  // after chunk i's weights come at most S-2 chunks of weight loads and one
  // of activation loads.
  static_assert((S - 2) * G::kJW + 2 * UPT <= 63, "vmcnt field");
  const int nch = c_end - c_begin;
  load_x(c_begin, xr[0]);
#pragma unroll
  for (int i = 0; i < S - 2; ++i) fetch_w(c_begin + i, i);
  load_x(c_begin + 1, xr[1]);
  fetch_w(c_begin + S - 2, S - 2);
  split_x(xb0, xr[0]);
  auto iteration = [&](auto pc, int i) {
    constexpr int p = decltype(pc)::value;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(sk_wait_imm((S - 2) * G::kJW + 2 * UPT));
    sk_barrier();
    load_x(c_begin + i + 2, xr[p]);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(c_begin + i + S - 1, (i + S - 1) % S);
    __builtin_amdgcn_sched_barrier(0);
    compute(i % S, xb0 + p * G::kXB);
    __builtin_amdgcn_sched_barrier(0);
    split_x(xb0 + (p ^ 1) * G::kXB, xr[p ^ 1]);
  };
  int i = 0;
  for (; i + 2 <= nch; i += 2) {
    iteration(std::integral_constant<int, 0>{}, i);
    iteration(std::integral_constant<int, 1>{}, i + 1);
  }
  if (i < nch) iteration(std::integral_constant<int, 0>{}, i);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  auto store = [&](int mt, int t, int i, float v) {
    const int n = n0 + 16 * t + r16, m = 16 * mt + 4 * s + i;
    if (n < N && m < M) C[(size_t)m * N + n] = v;
  };
  if (KG == 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) store(mt, t, i, acc[mt][t][i]);
    return;
  }
  // K split across workgroups: park this tile (float4 (mt*T + t) of thread
  // tid at index (mt*T + t) * 512 + tid, sc1 stores), count arrivals; the
  // last workgroup reads the KG tiles back and adds them in order kg =
  // 0..KG-1.  The loads of up to GB tiles are issued before any of them is
  // added: each load is a round trip to the level all XCDs share, so one
  // tile per round trip made the fix-up of a 16-way split take about 16 of
  // them.
  constexpr int NQ = MT * T;
  const CoherentTile tile_ws(reinterpret_cast<float4v*>(ws_part) + (size_t)(wg0 + tile * KG) * (NQ * 512),
                             (uint32_t)(KG * NQ * 512 * 16));
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t) tile_ws.store((uint32_t)kg * (NQ * 512) + (mt * T + t) * 512 + tid, acc[mt][t]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  __shared__ uint32_t is_last;
  if (tid == 0) {
    const uint32_t prev = __hip_atomic_fetch_add(&ws_cnt[ctr0 + tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = prev == (uint32_t)(KG - 1);
  }
  __syncthreads();
  if (!is_last) return;
  constexpr int GB = NQ >= kRingGatherF4 ? 1 : kRingGatherF4 / NQ;
  for (int g0 = 0; g0 < KG; g0 += GB) {
    float4v p[GB][MT][T];
#pragma unroll
    for (int gb = 0; gb < GB; ++gb) {
      const int g = g0 + gb;
      if (g < KG) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int t = 0; t < T; ++t) p[gb][mt][t] = tile_ws.load((uint32_t)g * (NQ * 512) + (mt * T + t) * 512 + tid);
      }
    }
#pragma unroll
    for (int gb = 0; gb < GB; ++gb) {
      const int g = g0 + gb;
      if (g < KG) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int t = 0; t < T; ++t) acc[mt][t] = g == 0 ? p[gb][mt][t] : acc[mt][t] + p[gb][mt][t];
      }
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) store(mt, t, i, acc[mt][t][i]);
  if (tid == 0) __hip_atomic_store(&ws_cnt[ctr0 + tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Ring geometry per format and weight tiles per wave (T): as many stages as
// fit in 160 KB of LDS beside the two split buffers, at most 4, at least 3.
template <class QF, int MT, int T>
struct RingCfg {
  typedef RingGeom<QF, MT, T> G;
  static constexpr int kFree = 160 * 1024 / 4 - 2 * G::kXB - 64;  // dwords (64 for the static LDS)
  static constexpr int kSLds = kFree / G::kStage, kSVm = 2 + (63 - 2 * G::kUPT) / G::kJW;  // LDS, vmcnt field
  static constexpr int kSMax = 4;  // deeper rings measured slower (fewer workgroups per CU)
  static constexpr int kS = kSLds < kSVm ? (kSLds < kSMax ? kSLds : kSMax) : (kSVm < kSMax ? kSVm : kSMax);
  static constexpr bool kOk = kS >= 3;
  static constexpr int kLds = (kS * G::kStage + 2 * G::kXB) * 4;
};

// Weight tiles per wave: the largest of 4, 2, 1 whose ring fits with at
// least 128 row groups (so a matrix spreads over the CUs with few K splits),
// else 1.
template <class QF, int MT>
int ring_t(uint32_t N) {
  if (RingCfg<QF, MT, 4>::kOk && N >= 128u * 512u) return 4;
  if (RingCfg<QF, MT, 2>::kOk && N >= 128u * 256u) return 2;
  return 1;
}

// Workgroups per row group (kg): up to about 256 workgroups in all, at
// least 2 chunks each where a row's whole K is at most 16 chunks, else 4,
// within the workspace; then longer K ranges (at least 8 chunks) where the
// launch keeps at least 128 workgroups, since each split adds a partial tile
// written and read back.  The choice depends on the job alone, so a grouped
// launch splits every job as its own launch would.
template <int MT, int T>
int ring_split(long tiles, uint32_t K, const nfhip::Workspace& ws) {
  const int NC = (int)(K / 64), min_chunks = NC <= 16 ? 2 : 4;
  int kg = 1;
  while (tiles * kg * 2 <= 256 && NC >= min_chunks * kg * 2 && tiles <= (long)ws.cnt_len &&
         (size_t)tiles * kg * 2 * MT * T * 512 * 4 <= ws.part_floats)
    kg *= 2;
  while (kg > 1 && NC / kg < 8 && tiles * (kg / 2) >= 128) kg /= 2;
  return kg;
}

// One launch for n jobs (n = 1: a single linear) over the same activations,
// each with the geometry and K split a launch of its own would get (so its
// output is bit-identical to that launch); hipErrorNotSupported if the
// jobs need different row tiles per wave or exceed the workspace.
template <class QF, int MT, int T>
hipError_t ring_group_t(const float* A, const nfhip::GemvJob* jobs, uint32_t n, uint32_t M, uint32_t K,
                        const nfhip::Workspace& ws, hipStream_t s) {
  typedef RingCfg<QF, MT, T> Cfg;
  if constexpr (!Cfg::kOk) {
    return hipErrorNotSupported;
  } else {
    RingGroup grp{};
    long wgs = 0, tiles = 0;
    bool split = false;
    for (uint32_t j = 0; j < n; ++j) {
      if (ring_t<QF, MT>(jobs[j].N) != T) return hipErrorNotSupported;
      const long t = ((long)jobs[j].N + 128 * T - 1) / (128 * T);
      const int kg = ring_split<MT, T>(t, K, ws);
      split = split || kg > 1;
      grp.W[j] = static_cast<const uint8_t*>(jobs[j].W);
      grp.C[j] = jobs[j].C;
      grp.N[j] = (int)jobs[j].N;
      grp.begin[j] = (int)wgs;
      grp.kg[j] = kg;
      grp.ctr[j] = (int)tiles;
      wgs += t * kg;
      tiles += t;
    }
    if (split && (tiles > (long)ws.cnt_len || (size_t)wgs * MT * T * 512 * 4 > ws.part_floats))
      return hipErrorNotSupported;
    for (int q = (int)n; q <= kSkGroupMax; ++q) grp.begin[q] = (int)wgs;
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&skinny_ring_kernel<QF, MT, T, Cfg::kS>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::kLds);
    if (attr != hipSuccess) return attr;
    skinny_ring_kernel<QF, MT, T, Cfg::kS><<<dim3((unsigned)wgs), dim3(512), Cfg::kLds, s>>>(
        A, grp.W[0], grp.N[0], grp.kg[0], grp.begin[1], grp.begin[2], grp.begin[3], (int)M, (int)K, grp.C[0],
        grp.ctr[0], ws.part, ws.cnt, grp);
    return hipGetLastError();
  }
}

template <class QF, int MT>
hipError_t ring_mt(const float* A, const nfhip::GemvJob* jobs, uint32_t n, uint32_t M, uint32_t K,
                   const nfhip::Workspace& ws, hipStream_t s) {
  const int t = ring_t<QF, MT>(jobs[0].N);
  if (t == 1) return ring_group_t<QF, MT, 1>(A, jobs, n, M, K, ws, s);
  if (t == 2) return ring_group_t<QF, MT, 2>(A, jobs, n, M, K, ws, s);
  if constexpr (MT == 4) return ring_group_t<QF, MT, 4>(A, jobs, n, M, K, ws, s);
  return hipErrorNotSupported;  // ring_serves() sends no such weights here
}

template <class QF>
hipError_t ring_dispatch(const float* A, const nfhip::GemvJob* jobs, uint32_t n, uint32_t M, uint32_t K,
                         const nfhip::Workspace& ws, hipStream_t s) {
  if (M <= 16) return ring_mt<QF, 1>(A, jobs, n, M, K, ws, s);
  if (M <= 32) return ring_mt<QF, 2>(A, jobs, n, M, K, ws, s);
  return ring_mt<QF, 4>(A, jobs, n, M, K, ws, s);
}

}  // namespace ring
}  // namespace nfk

namespace nfhip {

// Where f32 batches go to the ring kernel: two of its workgroups share a CU,
// which pays once the other kernel's would need a second round.  us in
// skinny.hip / here.  M = 64: Q4_0 50257x768 31.9 / 27.4, two 11008x4096 in a
// launch 69.9 / 63.0, but 4096x14336 35.6 / 40.9, 4096x4096 15.6 / 20.9; Q8_0
// 14336x4096 43.9 / 40.8, q, k and v of 4096, 1024 and 1024 rows at K = 4096
// 36.1 / 27.9, two 5632x2048 31.9 / 25.9, 16384x256 10.6 / 9.1, but 4096x1024
// 9.4 / 12.6, 768x768 6.5 / 9.4, 8192x256 6.3 / 9.7.  Up to 32 rows only where
// a row is a single 256-element chunk of the other kernel, whose ring then
// overlaps nothing: M = 8 Q8_0 24576x256 7.7 / 6.5, Q4_0 50257x256 9.4 / 7.7,
// but 16384x256 5.8 / 6.2 and 5.0 / 5.5, 65536x256 10.2 / 13.9 and 9.6 / 11.0,
// Q4_0 24576x512 7.4 / 7.7.
bool ring_serves(QFmt q, EType t, uint32_t M, uint32_t N, uint32_t K) {
  if (t != EType::F32 || M > 64) return false;
  if (M <= 32) return K <= 256 && N > 16384 && N < 65536;
  return N > 8192 || (q == QFmt::Q8_0 && (K > 2048 || (uint64_t)N * K > (4u << 20)));
}

hipError_t launch_skinny_ring(QFmt q, const void* A, const GemvJob* jobs, uint32_t n, uint32_t M, uint32_t K,
                              const Workspace& ws, hipStream_t s) {
  const float* a = static_cast<const float*>(A);
  return q == QFmt::Q4_0 ? nfk::ring::ring_dispatch<nfk::Q4_0>(a, jobs, n, M, K, ws, s)
                         : nfk::ring::ring_dispatch<nfk::Q8_0>(a, jobs, n, M, K, ws, s);
}

}  // namespace nfhip
