// First-order attention on gfx950 bf16 MFMA: the callers on either side of the double-backward.
//   attn_fwd_bf16     O and fp32 L = logsumexp        (fhog/triton_flash.py:12-133; L also replaces produce_L, :252-258)
//   attn_bwd_q_bf16   dQ                 Q-tiled      (fhog/triton_flash.py:201-220: P, dP, dS, dQ)
//   attn_bwd_k_bf16   dK, dV             K-tiled      (fhog/triton_flash.py:201-220: dV, dK)
// No atomics and nothing of shape (N_Q, N_K) in memory: like the double-backward, the backward recomputes
// S and dP once per tiling direction.
//
// A workgroup is 256 threads = 4 wave64 owning 128 stationary rows (queries, or keys in the K-tiled kernel);
// tiles of 32 streamed rows go through a two-stage LDS ring filled by direct global->LDS loads. First-level
// products are computed transposed (streamed rows = M, stationary rows = N), so a lane owns ONE stationary row
// and the soft-max statistics are per-lane scalars. The accumulator layout of such a product (lane = column,
// registers = streamed rows 8g + 4h + j) is, after rounding to bf16, already a valid B operand of the
// second-level MFMA whose contraction runs over the streamed rows: slot e of k-step t stands for streamed row
// 16t + 8(e/4) + 4h + e%4, and the A operand (the transposed value tile) is fetched from LDS with transposing
// reads that use the same row order. Second-level operands therefore never pass through LDS.
//
// What bounds them: vector and matrix instructions of a SIMD. Forward, 32 x 4096, d = 128, no mask: the matrix pipe is busy 43 %
// of the cycles and the VALU 48 %, and taking out the exponentials, the LDS reads or half of the staging moves the time by less
// than 5 %. Issuing the first level of a tile beside the second level of the tile before, each behind the other's
// elementwise work, measured equal (d = 64: +-3 %, d = 128: 2 % slower); fewer VALU instructions per block is what paid.
#include "fhog_bf16_blocks.h"

namespace fhog {
using namespace bf16k;
namespace {

// ---- forward -----------------------------------------------------------------------------------------
template <bool F16, int D, int MASK>
__global__ void __launch_bounds__(256, 2) attn_fwd_bf16(AttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int KK = D / 16, NC = D / 32, TILE = TS * 2 * D, STAGE = 2 * TILE;

  int bh, tile;
  // the forward keeps the tile-major order at every length: one slice after the other measures 2 % slower on 32 x 16384 rows
  if (!decode_block<MASK>((p.n_q + WG_ROWS - 1) / WG_ROWS, p.batch, MASK != MASK_NONE, MASK != MASK_NONE, bh, tile, MASK != MASK_NONE)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int q0 = tile * WG_ROWS, qw = q0 + 32 * wave, qi = qw + n;
  const int qr = min(qi, p.n_q - 1);  // queries past the end compute on a copy of the last row and store nothing
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb;
  const __bf16* src[2] = {(const __bf16*)p.k + koff, (const __bf16*)p.v + koff};

  bf16x8_t Qb[KK];
  load_resident<D>(Qb, (const __bf16*)p.q + qoff, p.stride_qn, qr, h);
  wait_vm0();
  const float c_scale_log2 = p.scale * kLog2e;

  int aoff[KK], troff[NC][2];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) aoff[kk] = tile_off<D>(n, 2 * kk + h);
#pragma unroll
  for (int cb = 0; cb < NC; cb++) {
    troff[cb][0] = tr_lane_off_acc<D>(cb, 0, lane);
    troff[cb][1] = tr_lane_off_acc<D>(cb, 1, lane);
  }
  float m = -INFINITY, l = 0.f;  // running maximum (log2 units) of the row; this lane's half of the row sum
  f32x16_t acc[1][NC];           // O^T: acc[0][cb][r] = (column 32cb + 8(r/4) + 4h + r%4, query qi)
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[0][cb] = f32x16_t{0};

  const StreamKeys<MASK> geo(p.mask_off, p.window, p.n_k);
  int j_begin, j_end;  // key tiles this workgroup visits
  geo.tile_range(q0, WG_ROWS, j_begin, j_end);
  Dma<D> dma;
  dma.init(p.stride_kn, wave, lane);
  const uint32_t ring_lds = lds_addr(smem);
  dma.template issue_all<2>(ring_lds, TILE, src, (int64_t)j_begin * TS * p.stride_kn, wave, p.n_k - j_begin * TS);
  dma_wait();
  __syncthreads();

  // Tile j in ring slot u. The slot is a constant: it goes into the offsets of the LDS reads.
  const auto step = [&](auto slot, int j) {
    constexpr int u = decltype(slot)::value;
    if (j + 1 < j_end) {
      const uint32_t dst = ring_lds + (u ^ 1) * STAGE;
      const int64_t adv = (int64_t)(j + 1) * TS * p.stride_kn;
      dma.template issue_all<2>(dst, TILE, src, adv, wave, p.n_k - (j + 1) * TS);
    }
    const int k0 = j * TS;
    const bool masked = geo.partial(k0, qw);  // wave-uniform: the block holds hidden keys (mask edge or tensor end)
    int lo = 0, hi = 0;                       // key k0 + 8g + 4h + e is visible iff lo <= 8g + e <= hi
    if (masked) keep_branch(), geo.limits(k0, qi, h, lo, hi);
    if (MASK == MASK_NONE || !geo.dead(k0, geo.first_row(qw, p.n_q))) {  // else every key of the tile is hidden from this wave
      const char* stage = smem + u * STAGE;
      fwd_block<F16, D>(stage, aoff, troff, Qb, masked, lo, hi, c_scale_log2, m, l, acc);
    }
    dma_wait();
    __syncthreads();
  };
  int j = j_begin;
  for (; j + 1 < j_end; j += 2) step(Slot<0>{}, j), step(Slot<1>{}, j + 1);
  if (j < j_end) step(Slot<0>{}, j);
  l += __shfl_xor(l, 32);
  const float inv = 1.f / l;
  if (qi >= p.n_q) return;
  __bf16* o = (__bf16*)p.o + qoff + (int64_t)qi * p.stride_qn;
#pragma unroll
  for (int cb = 0; cb < NC; cb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const f32x16_t& a = acc[0][cb];
      *reinterpret_cast<u32x2_t*>(o + 32 * cb + 8 * g + 4 * h) =
          pack4<F16>(a[4 * g] * inv, a[4 * g + 1] * inv, a[4 * g + 2] * inv, a[4 * g + 3] * inv);
    }
  if (h == 0) p.lse[(int64_t)bh * p.n_q + qi] = (m + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;  // v_log_f32 is log2
}

// ---- backward, Q-tiled: dQ, and d for the K-tiled kernel behind it ---------------------------------------
template <bool F16, int D, int MASK>
__global__ void __launch_bounds__(256, 2) attn_bwd_q_bf16(AttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int KK = D / 16, NC = D / 32, TILE = TS * 2 * D, STAGE = 2 * TILE;

  int bh, tile;
  if (!decode_block<MASK>((p.n_q + WG_ROWS - 1) / WG_ROWS, p.batch, MASK != MASK_NONE, p.tile_major_q != 0, bh, tile, MASK != MASK_NONE)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int q0 = tile * WG_ROWS, qw = q0 + 32 * wave, qi = qw + n;
  const int qr = min(qi, p.n_q - 1);  // queries past the end compute on a copy of the last row and store nothing
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb;
  const __bf16* src[2] = {(const __bf16*)p.k + koff, (const __bf16*)p.v + koff};

  bf16x8_t Qb[KK], dOb[KK];
  load_resident<D>(Qb, (const __bf16*)p.q + qoff, p.stride_qn, qr, h);
  load_resident<D>(dOb, (const __bf16*)p.dO + qoff, p.stride_qn, qr, h);
  const int64_t row = (int64_t)bh * p.n_q + qr;
  const float l_log2 = p.lse[row] * kLog2e;
  float dsum = 0.f;   // d_i = sum_c O_ic dO_ic: each lane takes half of its query's row
  {
    bf16x8_t Ob[KK];
    load_resident<D>(Ob, (const __bf16*)p.o + qoff, p.stride_qn, qr, h);
#pragma unroll
    for (int kk = 0; kk < KK; kk++)
#pragma unroll
      for (int e = 0; e < 8; e++) dsum = __builtin_fmaf(to_f32<F16>(Ob[kk][e]), to_f32<F16>(dOb[kk][e]), dsum);
    dsum += __shfl_xor(dsum, 32);
    if (h == 0 && qi < p.n_q) p.ws_d[row] = dsum;
  }
  wait_vm0();
  const float c_scale_log2 = p.scale * kLog2e;

  int aoff[KK], troff[NC][2];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) aoff[kk] = tile_off<D>(n, 2 * kk + h);
#pragma unroll
  for (int cb = 0; cb < NC; cb++) {
    troff[cb][0] = tr_lane_off_acc<D>(cb, 0, lane);
    troff[cb][1] = tr_lane_off_acc<D>(cb, 1, lane);
  }
  f32x16_t acc[1][NC];  // dQ^T
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[0][cb] = f32x16_t{0};

  const StreamKeys<MASK> geo(p.mask_off, p.window, p.n_k);
  int j_begin, j_end;  // key tiles this workgroup visits
  geo.tile_range(q0, WG_ROWS, j_begin, j_end);
  Dma<D> dma;
  dma.init(p.stride_kn, wave, lane);
  const uint32_t ring_lds = lds_addr(smem);
  dma.template issue_all<2>(ring_lds, TILE, src, (int64_t)j_begin * TS * p.stride_kn, wave, p.n_k - j_begin * TS);
  dma_wait();
  __syncthreads();

  // Tile j in ring slot u. The slot is a constant: it goes into the offsets of the LDS reads.
  const auto step = [&](auto slot, int j) {
    constexpr int u = decltype(slot)::value;
    if (j + 1 < j_end) {
      const uint32_t dst = ring_lds + (u ^ 1) * STAGE;
      const int64_t adv = (int64_t)(j + 1) * TS * p.stride_kn;
      dma.template issue_all<2>(dst, TILE, src, adv, wave, p.n_k - (j + 1) * TS);
    }
    const int k0 = j * TS;
    const bool masked = geo.partial(k0, qw);  // wave-uniform: the block holds hidden keys (mask edge or tensor end)
    int lo = 0, hi = 0;                       // key k0 + 8g + 4h + e is visible iff lo <= 8g + e <= hi
    if (masked) keep_branch(), geo.limits(k0, qi, h, lo, hi);
    if (MASK == MASK_NONE || !geo.dead(k0, geo.first_row(qw, p.n_q))) {
      const char* stage = smem + u * STAGE;
      bwd_q_block<F16, D>(stage, aoff, troff, Qb, dOb, masked, lo, hi, c_scale_log2, l_log2, dsum, acc);
    }
    dma_wait();
    __syncthreads();
  };
  int j = j_begin;
  for (; j + 1 < j_end; j += 2) step(Slot<0>{}, j), step(Slot<1>{}, j + 1);
  if (j < j_end) step(Slot<0>{}, j);
  if (qi >= p.n_q) return;
  __bf16* o = (__bf16*)p.dq + qoff + (int64_t)qi * p.stride_qn;
#pragma unroll
  for (int cb = 0; cb < NC; cb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const f32x16_t& a = acc[0][cb];
      *reinterpret_cast<u32x2_t*>(o + 32 * cb + 8 * g + 4 * h) =
          pack4<F16>(a[4 * g] * p.scale, a[4 * g + 1] * p.scale, a[4 * g + 2] * p.scale, a[4 * g + 3] * p.scale);
    }
}

// ---- backward, K-tiled: dK, dV (d = 64; at d = 128 attn_bwd_k_pc of fhog_bf16_pc.hip) ---------------------------------
template <bool F16, int D, int MASK>
__global__ void __launch_bounds__(256, 2) attn_bwd_k_bf16(AttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int KK = D / 16, NC = D / 32, TILE = TS * 2 * D;
  constexpr int STAT = 2 * TS * 4;         // L log2(e) and d of the 32 staged queries
  constexpr int STAGE = 2 * TILE + STAT;   // Q tile, dO tile, statistics

  int bh, tile;
  if (!decode_block<MASK>((p.n_k + WG_ROWS - 1) / WG_ROWS, p.batch, false, p.tile_major_k != 0, bh, tile, MASK != MASK_NONE)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int k0 = tile * WG_ROWS, kw = k0 + 32 * wave, kj = kw + n;
  const int kr = min(kj, p.n_k - 1);  // keys past the end compute on a copy of the last row and store nothing
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb;
  const __bf16* src[2] = {(const __bf16*)p.q + qoff, (const __bf16*)p.dO + qoff};
  const float* stat_src = (tid < TS ? p.lse : p.ws_d) + (int64_t)bh * p.n_q;

  bf16x8_t Kb[KK], Vb[KK];
  load_resident<D>(Kb, (const __bf16*)p.k + koff, p.stride_kn, kr, h);
  load_resident<D>(Vb, (const __bf16*)p.v + koff, p.stride_kn, kr, h);
  const float c_scale_log2 = p.scale * kLog2e;

  int aoff[KK], troff[NC][2];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) aoff[kk] = tile_off<D>(n, 2 * kk + h);
#pragma unroll
  for (int cb = 0; cb < NC; cb++) {
    troff[cb][0] = tr_lane_off_acc<D>(cb, 0, lane);
    troff[cb][1] = tr_lane_off_acc<D>(cb, 1, lane);
  }
  f32x16_t acc[2][NC];  // [0]: dK^T, [1]: dV^T
#pragma unroll
  for (int cb = 0; cb < NC; cb++) {
    acc[0][cb] = f32x16_t{0};
    acc[1][cb] = f32x16_t{0};
  }
  const StreamQueries<MASK> geo(p.mask_off, p.window, p.n_q);
  int t_begin, t_end;  // query tiles that hold a query seeing some key of this workgroup
  geo.tile_range(k0, WG_ROWS, t_begin, t_end);
  Dma<D> dma;
  dma.init(p.stride_qn, wave, lane);
  const uint32_t ring_lds = lds_addr(smem);
  float stat_reg = 0.f;  // threads 0..63: one statistic of the tile being staged
  // The statistic is loaded before the staging loads of a step and first touched at the end of the step, so the
  // wave never waits for it in between.
  auto load_stat = [&](int q_base) {
    if (tid < 2 * TS) stat_reg = *(global_f32_ptr)(stat_src + min(q_base + (tid & (TS - 1)), p.n_q - 1));
  };
  auto store_stat = [&](char* stage_base) {
    if (tid < 2 * TS) reinterpret_cast<float*>(stage_base + 2 * TILE)[tid] = (tid < TS) ? stat_reg * kLog2e : stat_reg;
  };
  {
    load_stat(t_begin * TS);
    const int64_t adv = (int64_t)t_begin * TS * p.stride_qn;
    dma.template issue_all<2>(ring_lds, TILE, src, adv, wave, p.n_q - t_begin * TS);
    wait_vm0();
    store_stat(smem);
  }
  __syncthreads();

  for (int j = t_begin; j < t_end; j++) {
    const int st = (j - t_begin) & 1;
    if (j + 1 < t_end) {
      load_stat((j + 1) * TS);
      const uint32_t dst = ring_lds + (st ^ 1) * STAGE;
      const int64_t adv = (int64_t)(j + 1) * TS * p.stride_qn;
      dma.template issue_all<2>(dst, TILE, src, adv, wave, p.n_q - (j + 1) * TS);
    }
    const int qb = j * TS;
    if (!geo.dead(qb, geo.first_row(kw, p.n_k))) {  // else no query of the tile sees a key of this wave
      const char* stage = smem + st * STAGE;
      bwd_k_block<F16, D>(geo, stage, aoff, troff, Kb, Vb, qb, kw, kj, h, c_scale_log2, acc);
    }
    if (j + 1 < t_end) {
      wait_vm0();
      store_stat(smem + (st ^ 1) * STAGE);
    }
    dma_wait();
    __syncthreads();
  }
  if (kj >= p.n_k) return;
  __bf16* odk = (__bf16*)p.dk + koff + (int64_t)kj * p.stride_kn;
  __bf16* odv = (__bf16*)p.dv + koff + (int64_t)kj * p.stride_kn;
#pragma unroll
  for (int cb = 0; cb < NC; cb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const f32x16_t& a = acc[0][cb];
      const f32x16_t& b = acc[1][cb];
      *reinterpret_cast<u32x2_t*>(odk + 32 * cb + 8 * g + 4 * h) =
          pack4<F16>(a[4 * g] * p.scale, a[4 * g + 1] * p.scale, a[4 * g + 2] * p.scale, a[4 * g + 3] * p.scale);
      *reinterpret_cast<u32x2_t*>(odv + 32 * cb + 8 * g + 4 * h) = pack4<F16>(b[4 * g], b[4 * g + 1], b[4 * g + 2], b[4 * g + 3]);
    }
}

template <auto Kernel>
hipError_t launch(unsigned grid, int smem, hipStream_t s, const AttnParams& p) {
  const hipError_t e = allow_dynamic_lds<Kernel>(smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(Kernel, dim3(grid), dim3(256), smem, s, p);
  return hipGetLastError();
}

template <bool F16, int D, int MASK>
hipError_t launch_attn_d(const AttnParams& p, int which, hipStream_t s) {
  constexpr int TILE = TS * 2 * D;
  switch (which) {
    case 0: return launch<attn_fwd_bf16<F16, D, MASK>>(grid_blocks((p.n_q + WG_ROWS - 1) / WG_ROWS, p.batch), 2 * 2 * TILE, s, p);
    case 1: return launch<attn_bwd_q_bf16<F16, D, MASK>>(grid_blocks((p.n_q + WG_ROWS - 1) / WG_ROWS, p.batch), 2 * 2 * TILE, s, p);
    default:
      if constexpr (D == 64)
        return launch<attn_bwd_k_bf16<F16, D, MASK>>(grid_blocks((p.n_k + WG_ROWS - 1) / WG_ROWS, p.batch), 2 * (2 * TILE + 2 * TS * 4), s, p);
      else
        return hipErrorInvalidValue;   // d = 128 is dispatched to the producer/consumer kernel before this point
  }
}

}  // namespace

// which: 0 forward, 1 backward Q-tiled (dQ), 2 backward K-tiled (dK, dV)
hipError_t launch_attn_bf16(const AttnParams& p, int which, hipStream_t s) {
  if (!bf16_shape_supported(p.n_q, p.n_k, p.d, p.causal)) return hipErrorInvalidValue;
  if (which == 2 && p.d == 128) return launch_attn_bwd_k_pc(p, s);   // one wave does not hold this sweep at d = 128
  const int mask = mask_mode(p);
#define FHOG_ATTN(F, DD)                                                            \
  (mask == MASK_NONE ? launch_attn_d<F, DD, MASK_NONE>(p, which, s)                 \
                     : mask == MASK_CAUSAL ? launch_attn_d<F, DD, MASK_CAUSAL>(p, which, s) : launch_attn_d<F, DD, MASK_BAND>(p, which, s))
  if (p.f16) return p.d == 128 ? FHOG_ATTN(true, 128) : FHOG_ATTN(true, 64);
  return p.d == 128 ? FHOG_ATTN(false, 128) : FHOG_ATTN(false, 64);
#undef FHOG_ATTN
}

}  // namespace fhog
