// Split-product double-backward of fp32 tensors for launches that leave most CUs idle: one output to a workgroup.
//
// A few heads of a few hundred tokens are as long as the longest chain of one wave: the tiles that it streams, one after the other, with nothing beside
// it on its SIMD. Passes 3 and 4 (fhog_split.hip) keep that at every fourth tile with eight products each, or at every second one with nine where
// the LDS does not hold four waves' tiles. Here dQ2, ddO, dK2 and dV2 have workgroups of their own, which compute S and ddS (and dP and E, where
// their output needs them) again: seven, five, seven and four products a tile, and LDS for the transposed operands of one output only,
// so that every launch has four waves (d = 128: two) on the same 32 rows. The work is a third more; it goes to CUs that have none.
//
// A wave takes every W-th streamed tile by itself. Its rows come straight into registers, two k-steps ahead, which is how the first level reads them; split
// into terms, those of the tensors that the second level contracts with are left in LDS of the wave's own for the transposing reads. So
// the sweep has no barrier; the partial results of the W waves are added through LDS in their order. At d = 128 a lane keeps 36 VGPRs (132 bytes) in
// scratch memory.
#include <type_traits>

#include "fhog_rules.h"
#include "fhog_split_util.h"

namespace fhog {
using namespace splitk;
namespace {

enum Output { kDQ2, kDDO, kDK2, kDV2 };

template <typename T, int D, int OUT>
struct Few {
  static constexpr bool KSIDE = OUT == kDK2 || OUT == kDV2, FULL = OUT == kDQ2 || OUT == kDK2;   // FULL: dP and E too
  static constexpr int NT = KSIDE ? 3 : 4;                     // streamed tensors: K, ddK, V, ddV | Q, ddQ, dO
  static constexpr int NR = FULL ? (KSIDE ? 4 : 3) : 2;        // stationary ones: Q, ddQ(, dO) | K, ddK(, V, ddV)
  static constexpr int FIRST = FULL ? 0 : 2, NS = OUT == kDV2 ? 1 : 2;   // left in LDS: tensors FIRST .. FIRST + NS - 1
  static constexpr int TENSOR = Terms<T>::N2 * TS * 2 * D, STAT = KSIDE ? 4 * TS * 4 : 0;
  static constexpr int BYTES = NS * TENSOR + STAT;             // of one wave
};

template <typename T, int D, int OUT, int MASK, int W>
__device__ __forceinline__ void run(const Params& p, char* smem, int id) {
  using S = Few<T, D, OUT>;
  constexpr bool KSIDE = S::KSIDE, FULL = S::FULL;
  constexpr int NT = S::NT, NR = S::NR, NS = S::NS, FIRST = S::FIRST, TENSOR = S::TENSOR, TILE = TS * 2 * D;
  constexpr int KK = D / 16, NC = D / 32, NF = Terms<T>::NF;
  static_assert(Terms<T>::NF == Terms<T>::N2 && Terms<T>::OFF2 == 0, "the terms of both levels are the same");

  const int tid = threadIdx.x, lane = tid & 63;
  const int ws = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int n_sta = KSIDE ? p.n_k : p.n_q, n_str = KSIDE ? p.n_q : p.n_k;
  int bh, tile;
  if (!decode_block<MASK>((n_sta + 31) / 32, p.batch, !KSIDE && MASK != MASK_NONE, KSIDE ? p.tile_major_k : p.tile_major, bh, tile, false, id)) return;
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb;
  const int64_t sta_ld = KSIDE ? p.stride_kn : p.stride_qn, str_ld = KSIDE ? p.stride_qn : p.stride_kn;
  const int rw = tile * 32, ri = rw + n, rr = min(ri, n_sta - 1);   // rows past the end compute on a copy of the last row and store nothing
  const T* src[NT];
  if constexpr (KSIDE) {
    src[0] = (const T*)p.q + qoff, src[1] = (const T*)p.ddq + qoff, src[2] = (const T*)p.dO + qoff;
  } else {
    src[0] = (const T*)p.k + koff, src[1] = (const T*)p.ddk + koff, src[2] = (const T*)p.v + koff, src[3] = (const T*)p.ddv + koff;
  }
  typename std::conditional<KSIDE, StreamQueries<MASK>, StreamKeys<MASK>>::type geo(p.mask_off, p.window, n_str);
  int t_begin, t_end;   // holds no tile that is dead to the rows
  geo.tile_range(rw, 32, t_begin, t_end);

  Chunk<T> ahead[2][NT];   // the next two k-steps of the lane's streamed row
  const auto load_step = [&](int t, int kk) {
    const int64_t off = (int64_t)min(t * TS + n, n_str - 1) * str_ld + 16 * kk + 8 * h;
#pragma unroll
    for (int x = 0; x < NT; x++) ahead[kk & 1][x] = load_chunk<T>(src[x] + off);
  };
  // statistics of the lane's streamed query
  const int64_t srow = (int64_t)bh * p.n_q;
  float stat_l = 0.f, stat_d = 0.f, stat_dd = 0.f, stat_b = 0.f;
  const auto load_stat = [&](int t) {
    const int64_t q = srow + min(t * TS + n, p.n_q - 1);
    stat_l = p.lse[q], stat_dd = p.ws_dd[q];
    if (FULL) stat_d = p.ws_d[q], stat_b = p.ws_b[q];
  };
  if (t_begin + ws < t_end) {
    load_step(t_begin + ws, 0), load_step(t_begin + ws, 1);
    if (KSIDE) load_stat(t_begin + ws);
  }

  const T* const sta[4] = {KSIDE ? (const T*)p.k + koff : (const T*)p.q + qoff, KSIDE ? (const T*)p.ddk + koff : (const T*)p.ddq + qoff,
                           KSIDE ? (const T*)p.v + koff : (const T*)p.dO + qoff, (const T*)p.ddv + koff};
  Resident<T, D> res[NR];
#pragma unroll
  for (int x = 0; x < NR; x++) res[x].load(sta[x] + (int64_t)rr * sta_ld, h);
  const int64_t row = srow + rr;   // dQ2, ddO
  float l_log2 = 0.f, dsum = 0.f, dd = 0.f, kc = 0.f;
  if constexpr (!KSIDE) {
    l_log2 = p.lse[row] * kLog2e, dd = p.ws_dd[row];
    if constexpr (FULL) dsum = p.ws_d[row], kc = __builtin_fmaf(dd, dsum, p.ws_b[row]);
  }
  const float c_scale_log2 = p.scale * kLog2e;

  int troff[NC][2];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) troff[cb][0] = tr_lane_off_acc<D>(cb, 0, lane), troff[cb][1] = tr_lane_off_acc<D>(cb, 1, lane);
  f32x16_t acc[NC];   // lane = stationary row, registers = columns
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[cb] = f32x16_t{0};

  char* const own = smem + ws * S::BYTES;
  float* const stat = reinterpret_cast<float*>(own + NS * TENSOR);   // L log2(e), -d, dd, -(dd d + b) of the 32 queries
  for (int t = t_begin + ws; t < t_end; t += W) {
    const int s0 = t * TS;
    f32x16_t s = {0}, dds = {0}, dp = {0}, e = {0};
    if constexpr (KSIDE) {
      stat[(h ? 2 * TS : 0) + n] = h ? stat_dd : stat_l * kLog2e;
      if constexpr (FULL) stat[(h ? 3 * TS : TS) + n] = h ? -__builtin_fmaf(stat_dd, stat_d, stat_b) : -stat_d;
      load_stat(t + W < t_end ? t + W : t);
      if constexpr (FULL) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const f32x4_t md4 = *reinterpret_cast<const f32x4_t*>(stat + 1 * TS + 8 * g + 4 * h);
          const f32x4_t mk4 = *reinterpret_cast<const f32x4_t*>(stat + 3 * TS + 8 * g + 4 * h);
#pragma unroll
          for (int i = 0; i < 4; i++) dp[4 * g + i] = md4[i], e[4 * g + i] = mk4[i];
        }
      }
    } else if constexpr (FULL) {   // u = dP - d and E' = E - (dd d + b) come straight from accumulators that start at the row constants
#pragma unroll
      for (int r = 0; r < 16; r++) dp[r] = -dsum, e[r] = -kc;
    }
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
      bf16x8_t a[NF], r0[NF], r1[NF], r2[NF], r3[NF];
      res[0].terms(kk, r0), res[1].terms(kk, r1);
      if constexpr (FULL) res[2].terms(kk, r2), res[NR - 1].terms(kk, r3);
      // the terms of tensor x, left in LDS where the second level wants them; split with ANY from the third tensor on, as in fhog_split.hip
      const auto streamed = [&](auto xc) {
        constexpr int x = decltype(xc)::value;
        chunk_terms<T, true, (x >= 2)>(ahead[kk & 1][x], a);
        if constexpr (x >= FIRST && x < FIRST + NS) {
#pragma unroll
          for (int q = 0; q < NF; q++) *reinterpret_cast<bf16x8_t*>(own + (x - FIRST) * TENSOR + q * TILE + tile_off<D>(n, 2 * kk + h)) = a[q];
        }
      };
      streamed(std::integral_constant<int, 0>{});
      s = mma1<T>(s, a, r0);                                    // K Q^T | Q K^T
      dds = mma1<T>(dds, a, r1);                                // K ddQ^T | Q ddK^T
      streamed(std::integral_constant<int, 2>{});
      if constexpr (FULL) dp = mma1<T>(dp, a, r2);              // V dO^T | dO V^T
      if constexpr (FULL && KSIDE) e = mma1<T>(e, a, r3);       // dO ddV^T
      streamed(std::integral_constant<int, 1>{});
      dds = mma1<T>(dds, a, r0);                                // + ddK Q^T | ddQ K^T
      if constexpr (!KSIDE) streamed(std::integral_constant<int, 3>{});
      if constexpr (FULL && !KSIDE) e = mma1<T>(e, a, r2);      // ddV dO^T
      load_step(kk + 2 < KK ? t : t + W, (kk + 2) % KK);        // past the last tile: its last row again
      __builtin_amdgcn_sched_barrier(0);
    }
    f32x16_t pv;
#pragma unroll
    for (int g = 0; g < 4; g++) {
      f32x4_t l4 = {l_log2, l_log2, l_log2, l_log2};
      if constexpr (KSIDE) l4 = *reinterpret_cast<const f32x4_t*>(stat + 8 * g + 4 * h);
#pragma unroll
      for (int i = 0; i < 4; i++) pv[4 * g + i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * g + i], c_scale_log2, -l4[i]));
    }
    if (geo.partial(s0, rw)) {   // wave-uniform: the block holds hidden pairs (mask edge or tensor end)
      int lo, hi;
      geo.limits(s0, ri, h, lo, hi);
      keep_branch();
#pragma unroll
      for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
    }
#pragma unroll
    for (int g = 0; g < 4; g++) {
      f32x4_t dd4 = {dd, dd, dd, dd};
      if constexpr (KSIDE) dd4 = *reinterpret_cast<const f32x4_t*>(stat + 2 * TS + 8 * g + 4 * h);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = 4 * g + i;
        dds[r] = pv[r] * __builtin_fmaf(dds[r], p.scale, -dd4[i]);   // ddP = P w
        if constexpr (FULL) {
          s[r] = pv[r] * dp[r];                                       // dS = P u (scale applied to the accumulator at the end)
          e[r] = __builtin_fmaf(pv[r], e[r], dds[r] * dp[r]);         // dS' = P E' + ddP u
        }
      }
    }
    if constexpr (FULL) {
      second_level<T, D>(acc, own + TENSOR, troff, s);   // dQ2 += dS ddK | dK2 += dS^T ddQ
      second_level<T, D>(acc, own, troff, e);            // dQ2 += dS' K | dK2 += dS'^T Q
    } else {
      if constexpr (!KSIDE) second_level<T, D>(acc, own + TENSOR, troff, pv);   // ddO += P ddV
      second_level<T, D>(acc, own, troff, dds);                                 // ddO += ddP V | dV2 += ddP^T dO
    }
  }

  // the waves add their partial results in the order of ws; the first one holds the sum
  float* const xch = reinterpret_cast<float*>(smem) + lane;
  __syncthreads();   // the tiles are no longer read
  if (ws > 0) {
#pragma unroll
    for (int cb = 0; cb < NC; cb++)
#pragma unroll
      for (int r = 0; r < 16; r++) xch[((ws - 1) * NC * 16 + cb * 16 + r) * 64] = acc[cb][r];
  }
  __syncthreads();
  if (ws > 0) return;
#pragma unroll
  for (int o = 1; o < W; o++)
#pragma unroll
    for (int cb = 0; cb < NC; cb++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[cb][r] += xch[((o - 1) * NC * 16 + cb * 16 + r) * 64];
  if (ri >= n_sta) return;
  T* const out = (T*)(OUT == kDQ2 ? p.dq2 : OUT == kDDO ? p.ddo : OUT == kDK2 ? p.dk2 : p.dv2) + (KSIDE ? koff : qoff) + (int64_t)ri * sta_ld;
  store_rows<T, D>(out, acc, FULL ? p.scale : 1.f, h);
}

// Workgroups of dQ2, dK2, ddO and dV2, in this order: gq of the query side's outputs each, gk of the key side's
template <typename T, int D, int MASK, int W>
__global__ void __launch_bounds__(64 * W, 1) split_few(Params p, int gq, int gk) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  int id = blockIdx.x;
  if (id < gq) return run<T, D, kDQ2, MASK, W>(p, smem, id);
  if ((id -= gq) < gk) return run<T, D, kDK2, MASK, W>(p, smem, id);
  if ((id -= gk) < gq) return run<T, D, kDDO, MASK, W>(p, smem, id);
  run<T, D, kDV2, MASK, W>(p, smem, id - gq);
}

template <int D, int MASK>
hipError_t launch(const Params& p, int sides, hipStream_t s) {
  constexpr int W = D == 128 ? 2 : 4;
  constexpr int smem = W * (Few<float, D, kDK2>::BYTES > Few<float, D, kDQ2>::BYTES ? Few<float, D, kDK2>::BYTES : Few<float, D, kDQ2>::BYTES);
  static_assert(smem <= 160 * 1024 && smem >= (W - 1) * (D / 32) * 16 * 64 * 4, "the waves' tiles have to fit the LDS, and the exchange in their place");
  const hipError_t e = allow_dynamic_lds<split_few<float, D, MASK, W>>(smem);
  if (e != hipSuccess) return e;
  const unsigned gq = sides & 1 ? grid_blocks((p.n_q + 31) / 32, p.batch) : 0, gk = sides & 2 ? grid_blocks((p.n_k + 31) / 32, p.batch) : 0;
  hipLaunchKernelGGL((split_few<float, D, MASK, W>), dim3(2 * (gq + gk)), dim3(64 * W), smem, s, p, (int)gq, (int)gk);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_split_few(const Params& p, int sides, hipStream_t s) {
#define FHOG_FEW(D) (p.causal ? launch<D, MASK_BAND>(p, sides, s) : launch<D, MASK_NONE>(p, sides, s))
  switch (p.d) {
    case 32: return FHOG_FEW(32);
    case 64: return FHOG_FEW(64);
    case 128: return FHOG_FEW(128);
    default: return hipErrorInvalidValue;
  }
#undef FHOG_FEW
}

}  // namespace fhog
