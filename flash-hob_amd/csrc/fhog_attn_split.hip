// First-order attention on split products (fhog_split_util.h): contractions of fp32 accuracy on the 16-bit matrix
// instructions. Forward (O and the fp32 log-sum-exp L, online soft-max; fhog/triton_flash.py:12-133, 252-258) and backward
// (dQ; dK and dV; the arithmetic of fhog/triton_flash.py:201-220 without the (batch, N_Q, N_K) tensors and without
// atomics). Serves fp32 tensors and d = 32, the shapes the 16-bit kernels of fhog_attn.hip do not take.
//
// Same shape as the double-backward kernels of fhog_split.hip: a workgroup of 4 wave64 owns 32 stationary rows per wave
// (queries; keys in the K-tiled backward) with their operands in registers as bf16 terms, the other side streams through
// LDS in 32-row tiles that are split once per workgroup. A lane owns ONE stationary row: in the forward the running maximum,
// the running sum and the rescaling factor of a query are per-lane scalars. Two terms per fp32 operand less than the
// double-backward needs leave room for the terms of d = 128 (one wave per SIMD); only dK, dV on fp32 tensors there does not quite
// fit and keeps 42 to 118 VGPRs of a lane in scratch memory under a mask or with two waves on the same rows.
// Small launches (WS = 2 or 4) put WS waves on the same 32 rows: each takes every WS-th streamed tile, and the partial
// results are merged through LDS in a fixed order. dQ and dK, dV share a launch unless each fills the GPU (launch_bwd).
#include <type_traits>

#include "fhog_rules.h"
#include "fhog_split_util.h"

namespace fhog {
using namespace splitk;
namespace {

constexpr int MODE_FWD = 0, MODE_BWD_Q = 1, MODE_BWD_K = 2;

// Workgroups on a CU that the registers are to leave room for. At d = 64 two keep a SIMD busy where one waits (for LDS operands, the
// splitting, a barrier): 256 registers each, short of 2 (no mask) and 8 where dQ and dK, dV share a launch. us, one -> two, fp32 causal 32 x 2048 | no mask 64 x 2048: forward 146 -> 128 |
// 410 -> 368, dQ 193 -> 158 | 528 -> 495, dK, dV 238 -> 209 | 783 -> 648. At d = 128 so does the forward (TWO), without the second stage of
// the ring and with the query's numbers instead of their terms; worth it in launches with work for two on every CU (launch_fwd). At d = 32 also with
// waves on the same rows: first backward of fp32 causal 16 x 1024, four of them, 53 us with two workgroups and 66 with one.
template <typename T, int D, int WS, bool TWO>
constexpr int min_workgroups = (WS > 1 && D > 32) || (sizeof(T) * D > 256 && !TWO) ? 1 : 2;

// Stages of the ring. With a wave split the WS tiles of a step take the room of the second one.
template <int WS, bool TWO>
constexpr int n_buffers = WS == 1 && !TWO ? 2 : 1;

// OWN_D: dK, dV without the sweep for dQ before it; pairs: as decode_block takes it
template <typename T, int D, int MODE, int MASK, int WS, bool OWN_D, bool TWO = false>
__device__ __forceinline__ void attn_run(const AttnParams& p, char* smem, int id, bool pairs) {
  constexpr bool KSIDE = MODE == MODE_BWD_K;
  // split_pair: two waves of fp32 tensors on a SIMD run faster without the dot products (dK, dV causal 32 x 2048, d = 64 231 -> 217 us), the VALU-bound ones of
  // 16-bit tensors with them (bf16 causal 64 x 1024, d = 32 86.5 against 89.3 us for both first-order passes)
  constexpr bool DOT = sizeof(T) == 2 || D == 32;
  constexpr int NR = MODE == MODE_FWD ? 1 : 2;             // stationary tensors: Q | Q, dO | K, V
  constexpr int KK = D / 16, NC = D / 32, NF = Terms<T>::NF;
  using Stage = Stager<T, D, 2, true, 0, DOT>;                     // streamed tensors: K, V | Q, dO
  constexpr int TENSOR = Stage::PLANES * Stage::TILE;
  constexpr int STAT = KSIDE ? 2 * TS * 4 : 0;             // L log2(e), -d of the 32 staged queries
  constexpr int STAGE = Stage::BYTES + STAT;
  constexpr int NBUF = n_buffers<WS, TWO>;
  constexpr int nw = 4 / WS, ROWS = 32 * nw;
  constexpr bool RAW = TWO;
  // the next tile is split and written to LDS behind the MFMAs of this one: forward of fp32, d = 64, no mask 64 x 2048 383 -> 371 us
  constexpr bool INTERLEAVED = MODE == MODE_FWD && sizeof(T) == 4 && D == 64 && WS == 1;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wv / WS, ws = wv % WS;   // row group of the wave, and which of the streamed tiles of a step it takes
  const int n = lane & 31, h = lane >> 5;
  const int n_sta = KSIDE ? p.n_k : p.n_q, n_str = KSIDE ? p.n_q : p.n_k;
  int bh, tile;
  if (!decode_block<MASK>((n_sta + ROWS - 1) / ROWS, p.batch, !KSIDE && MASK != MASK_NONE, MASK != MASK_NONE, bh, tile, pairs, id)) return;
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb;
  const int64_t sta_ld = KSIDE ? p.stride_kn : p.stride_qn, str_ld = KSIDE ? p.stride_qn : p.stride_kn;
  const int r0 = tile * ROWS, rw = r0 + 32 * group, ri = rw + n;
  const int rr = min(ri, n_sta - 1);         // rows past the end compute on a copy of the last row and store nothing
  const T* const src[2] = {KSIDE ? (const T*)p.q + qoff : (const T*)p.k + koff, KSIDE ? (const T*)p.dO + qoff : (const T*)p.v + koff};

  typename std::conditional<KSIDE, StreamQueries<MASK>, StreamKeys<MASK>>::type geo(p.mask_off, p.window, n_str);
  int t_begin, t_end;
  geo.tile_range(r0, ROWS, t_begin, t_end);

  const int64_t srow = (int64_t)bh * p.n_q;
  Stage st[WS];
  // dK, dV: L and d of the staged queries. OWN_D: d_i = sum_c O_ic dO_ic is taken here, by the threads that stage the row of dO.
  constexpr int DO0 = Stage::RPT / Stage::XPI;                     // first chunk of dO among the chunks that a thread stages
  float stat_reg[WS] = {};
  Chunk<T> o_reg[WS][KSIDE && OWN_D ? Stage::RPT : 1];
  const auto fetch = [&](int t) {
#pragma unroll
    for (int g = 0; g < WS; g++) {
      const int row0 = min((t + g) * TS, n_str - 1);                // a tile past the end is never computed on
      st[g].fetch(src, str_ld, row0, n_str, tid);
      if (KSIDE && tid < (OWN_D ? 1 : 2) * TS) stat_reg[g] = (tid < TS ? p.lse : p.ws_d)[srow + min(row0 + (tid & 31), p.n_q - 1)];
      if constexpr (KSIDE && OWN_D) {
#pragma unroll
        for (int i = 0; i < Stage::RPT; i++)
          o_reg[g][i] = load_chunk<T>((const T*)p.o + qoff + (int64_t)min(row0 + Stage::row_of(DO0 + i, tid), p.n_q - 1) * str_ld + 8 * (tid % Stage::CPR));
      }
    }
  };
  const auto publish = [&](int buf) {
#pragma unroll
    for (int g = 0; g < WS; g++) {
      char* stage = smem + (buf * WS + g) * STAGE;
      st[g].publish(stage, tid);
      float* const stat = reinterpret_cast<float*>(stage + Stage::BYTES);
      if (KSIDE && tid < (OWN_D ? 1 : 2) * TS) stat[tid] = tid < TS ? stat_reg[g] * kLog2e : -stat_reg[g];
      if constexpr (KSIDE && OWN_D) {
#pragma unroll
        for (int i = 0; i < Stage::RPT; i++) {
          float d = 0.f;
#pragma unroll
          for (int e = 0; e < 8; e++) d = __builtin_fmaf(chunk_elem(o_reg[g][i], e), chunk_elem(st[g].c[DO0 + i], e), d);
#pragma unroll
          for (int m = 1; m < Stage::CPR; m *= 2) d += __shfl_xor(d, m);
          // two tensors in a round of threads: the second half of them holds dO
          if (tid % Stage::CPR == 0 && (Stage::XPI == 1 || tid >= 128)) stat[TS + Stage::row_of(DO0 + i, tid)] = -d;
        }
      }
    }
  };
  if (t_begin < t_end) fetch(t_begin);

  bf16x8_t res[NR][KK][NF];
  Chunk<T> raw[KK];                // RAW: the fp32 numbers of a query, split again for every tile
  if constexpr (RAW) {
#pragma unroll
    for (int kk = 0; kk < KK; kk++) raw[kk] = load_chunk<T>((const T*)p.q + qoff + (int64_t)rr * sta_ld + 16 * kk + 8 * h);
  } else {
    load_resident_terms<T, D>(res[0], KSIDE ? (const T*)p.k + koff : (const T*)p.q + qoff, sta_ld, rr, h);
  }
  if constexpr (MODE != MODE_FWD)
    load_resident_terms<T, D>(res[NR - 1], KSIDE ? (const T*)p.v + koff : (const T*)p.dO + qoff, sta_ld, rr, h);
  const int64_t row = srow + rr;   // Q-tiled kernels
  float l_log2 = 0.f, dsum = 0.f;
  if constexpr (MODE == MODE_BWD_Q) {
    // d_i = sum_c O_ic dO_ic, for this sweep and (through the workspace) for the K-tiled one behind it: each lane takes
    // half of its query's row
    l_log2 = p.lse[row] * kLog2e;
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
      const Chunk<T> o = load_chunk<T>((const T*)p.o + qoff + (int64_t)rr * sta_ld + 16 * kk + 8 * h);
      const Chunk<T> g = load_chunk<T>((const T*)p.dO + qoff + (int64_t)rr * sta_ld + 16 * kk + 8 * h);
#pragma unroll
      for (int e = 0; e < 8; e++) dsum = __builtin_fmaf(chunk_elem(o, e), chunk_elem(g, e), dsum);
    }
    dsum += __shfl_xor(dsum, 32);
    if (h == 0 && ri < p.n_q && ws == 0) p.ws_d[row] = dsum;
  }
  const float c_scale_log2 = p.scale * kLog2e;

  int aoff[KK], troff[NC][2];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) aoff[kk] = tile_off<D>(n, 2 * kk + h);
#pragma unroll
  for (int cb = 0; cb < NC; cb++) troff[cb][0] = tr_lane_off_acc<D>(cb, 0, lane), troff[cb][1] = tr_lane_off_acc<D>(cb, 1, lane);

  float m = -INFINITY, l = 0.f;    // forward: running maximum (log2 units) of the row; this lane's half of the row sum
  f32x16_t acc0[NC], acc1[NC];     // O | dQ | dK, dV: lane = stationary row, registers = columns
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc0[cb] = f32x16_t{0}, acc1[cb] = f32x16_t{0};

  // INTERLEAVED: the first level of a tile; LDS operands are read behind the MFMAs of the k-step before, and behind(slot, slots) is what
  // else is to be done behind MFMA `slot`. The fences hold the order.
  const auto first_level = [&](const char* stage, f32x16_t& s, auto behind) {
    constexpr TermPairs<NF, NF> kPairs{};
    constexpr int P = kPairs.n;
    bf16x8_t a[2][NF];
    read_terms<T, Stage::TILE>(stage, aoff[0], a[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < KK; kk++)
#pragma unroll
      for (int i = 0; i < P; i++) {
        s = mfma<false>(a[kk & 1][kPairs.a[i]], res[0][kk][kPairs.b[i]], s);
        if (i == 0 && kk + 1 < KK) read_terms<T, Stage::TILE>(stage, aoff[kk + 1], a[(kk + 1) & 1]);
        behind(P * kk + i, P * KK);
        __builtin_amdgcn_sched_barrier(0);
      }
    asm volatile("" : "+v"(s));   // holds the products in front of the branches that follow: the compiler sinks them to the use of their sum
  };

  const auto block = [&](const char* stage, int s0, auto behind) {
    const float* stat = reinterpret_cast<const float*>(stage + Stage::BYTES);
    f32x16_t s = {0}, dp = {0};
    if constexpr (MODE == MODE_BWD_Q) {   // u = dP - d comes straight from an accumulator that starts at -d
#pragma unroll
      for (int r = 0; r < 16; r++) dp[r] = -dsum;
    } else if constexpr (KSIDE) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x4_t md4 = *reinterpret_cast<const f32x4_t*>(stat + TS + 8 * g + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; i++) dp[4 * g + i] = md4[i];
      }
    }
    if constexpr (INTERLEAVED) {
      first_level(stage, s, behind);
    } else {
#pragma unroll
      for (int kk = 0; kk < KK; kk++) {
        bf16x8_t a[NF];
        read_terms<T, Stage::TILE>(stage, aoff[kk], a);
        if constexpr (RAW) {
          bf16x8_t q[NF];
          // splitting is to happen here, tile after tile: hoisted out of the sweep, the terms would be spilled
          asm volatile("" : "+v"(raw[kk].v[0]), "+v"(raw[kk].v[1]));
          chunk_terms<T, true, true, DOT>(raw[kk], q);
          s = mma1<T>(s, a, q);
        } else {
          s = mma1<T>(s, a, res[0][kk]);                        // K Q^T | Q K^T
        }
        if constexpr (MODE != MODE_FWD) {
          bf16x8_t g[NF];
          read_terms<T, Stage::TILE>(stage + TENSOR, aoff[kk], g);
          dp = mma1<T>(dp, g, res[NR - 1][kk]);                 // V dO^T | dO V^T
        }
      }
    }
    const bool masked = geo.partial(s0, rw);   // wave-uniform: the block holds hidden pairs (mask edge or tensor end)
    int lo = 0, hi = 0;
    if (masked) keep_branch(), geo.limits(s0, ri, h, lo, hi);
    f32x16_t pv;
    if constexpr (MODE == MODE_FWD) {
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] *= c_scale_log2;      // before the maximum is taken: any sign of the scale
      if (masked) {
        keep_branch();
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = in_limits(r, lo, hi) ? s[r] : -INFINITY;
      }
      float tmax = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
      for (int r = 3; r < 15; r += 2) tmax = fmaxf(fmaxf(tmax, s[r]), s[r + 1]);
      tmax = fmaxf(tmax, s[15]);
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32));   // the other half of the wave holds the other 16 keys of the row
      const float m_new = fmaxf(m, tmax);
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;   // a row that has seen no key yet keeps its state
      const float alpha = __builtin_amdgcn_exp2f(m - m_ref);
      float rs = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        pv[r] = __builtin_amdgcn_exp2f(s[r] - m_ref);
        rs += pv[r];
      }
      l = __builtin_fmaf(l, alpha, rs);
      if (__builtin_amdgcn_ballot_w64(m_new > m) != 0) {   // rescale only when some row's maximum moved
#pragma unroll
        for (int cb = 0; cb < NC; cb++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc0[cb][r] *= alpha;
      }
      m = m_new;
      if constexpr (INTERLEAVED) {
        SecondLevel<T, D> second{troff[0][0], troff[0][1]};
        second.start(stage + TENSOR, pv);
        second.template run<false>(acc0, stage + TENSOR, pv, stage, pv, [](int) {});   // O += P V
      } else {
        second_level<T, D, DOT>(acc0, stage + TENSOR, troff, pv);
      }
    } else {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        f32x4_t l4 = {l_log2, l_log2, l_log2, l_log2};
        if constexpr (KSIDE) l4 = *reinterpret_cast<const f32x4_t*>(stat + 8 * g + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; i++) pv[4 * g + i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * g + i], c_scale_log2, -l4[i]));
      }
      if (masked) {
        keep_branch();
#pragma unroll
        for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
      }
#pragma unroll
      for (int r = 0; r < 16; r++) dp[r] *= pv[r];            // dS = P (dP - d) (scale applied to the accumulators at the end)
      second_level<T, D, DOT>(acc0, stage, troff, dp);             // dQ += dS K | dK += dS^T Q
      if constexpr (KSIDE) second_level<T, D, DOT>(acc1, stage + TENSOR, troff, pv);   // dV += P^T dO
    }
  };

  if (t_begin < t_end) publish(0);
  if (INTERLEAVED && t_begin < t_end) fetch(t_begin + 1);
  __syncthreads();
  // Without a mask only waves whose rows all lie past the end of the tensor see nothing. fp32, d = 128: a test for them in the loop has the compiler spill
  // what a wave keeps (dK, dV 42 VGPRs), so they have a loop of their own; with two waves on the same rows they compute on copies of the last row. First-order
  // passes, us, no test | the test | two loops: 32 x 1024 430 | 459 | 425, 64 x 2048 3280 | 3554 | 3213, 2000 | 900 rows 432 | 501 | 423, 128 x 300 249 |
  // 264 | 233; two waves 16 x 300 84.3 | 85.2 | 86.3, 4 x 1024 228 | 231 | 229. At d = 32 the test is the faster (bf16 16 x 4096 412 | 420).
  constexpr bool NO_TEST = MASK == MASK_NONE && is_raw<T, D>;
  const auto sweep = [&](auto has_rows) {
    const auto works = [&](int s0) { return NO_TEST ? decltype(has_rows)::value : !geo.dead(s0, geo.first_row(rw, n_sta)); };
    for (int t = t_begin; t < t_end; t += WS) {
      const int buf = NBUF == 2 ? (t - t_begin) & 1 : 0;
      if constexpr (INTERLEAVED) {
        // The rows of the tile after this one came in during the step before; behind the last tile they are copies of the last row.
        char* const next = smem + (buf ^ 1) * STAGE;
        const int s0 = t * TS, row0 = min(s0 + 2 * TS, n_str - 1);
        if (works(s0)) {
          block(smem + buf * STAGE, s0, [&](int slot, int slots) {
            st[0].publish_at(next, tid, slot, slots, [&](int i) { st[0].fetch_chunk(i, src, str_ld, row0, n_str, tid); });
          });
        } else {
          publish(buf ^ 1);
          fetch(t + 2);
        }
        __syncthreads();
        continue;
      }
      const bool more = t + WS < t_end;
      if (more) fetch(t + WS);
      const int s0 = (t + ws) * TS;
      if ((WS == 1 || t + ws < t_end) && works(s0)) block(smem + (buf * WS + ws) * STAGE, s0, [](int, int) {});
      if (NBUF == 1) __syncthreads();   // the tiles are no longer read
      if (more) publish(NBUF == 2 ? buf ^ 1 : 0);
      __syncthreads();
    }
  };
  if (NO_TEST && WS == 1 && rw >= n_sta) sweep(std::false_type{});
  else sweep(std::true_type{});

  if constexpr (WS > 1) {
    // the WS waves of a row group merge their partial results in the order of ws; the wave with ws == 0 holds the outcome
    constexpr int VALS = (KSIDE ? 2 : 1) * NC * 16 + (MODE == MODE_FWD ? 2 : 0);
    float* const xch = reinterpret_cast<float*>(smem) + lane;
    if (ws > 0) {
      float* dst = xch + (group * (WS - 1) + ws - 1) * VALS * 64;
#pragma unroll
      for (int cb = 0; cb < NC; cb++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          dst[(cb * 16 + r) * 64] = acc0[cb][r];
          if constexpr (KSIDE) dst[((NC + cb) * 16 + r) * 64] = acc1[cb][r];
        }
      if constexpr (MODE == MODE_FWD) dst[(VALS - 2) * 64] = m, dst[(VALS - 1) * 64] = l;
    }
    __syncthreads();
    if (ws > 0) return;
#pragma unroll
    for (int o = 1; o < WS; o++) {
      const float* from = xch + (group * (WS - 1) + o - 1) * VALS * 64;
      float mine = 1.f, theirs = 1.f;
      if constexpr (MODE == MODE_FWD) {
        const float mo = from[(VALS - 2) * 64], m_new = fmaxf(m, mo), m_ref = m_new == -INFINITY ? 0.f : m_new;
        mine = __builtin_amdgcn_exp2f(m - m_ref), theirs = __builtin_amdgcn_exp2f(mo - m_ref);
        l = __builtin_fmaf(l, mine, from[(VALS - 1) * 64] * theirs);
        m = m_new;
      }
#pragma unroll
      for (int cb = 0; cb < NC; cb++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          acc0[cb][r] = __builtin_fmaf(from[(cb * 16 + r) * 64], theirs, acc0[cb][r] * mine);
          if constexpr (KSIDE) acc1[cb][r] += from[((NC + cb) * 16 + r) * 64];
        }
    }
  }

  if constexpr (MODE == MODE_FWD) l += __shfl_xor(l, 32);
  if (ri >= n_sta) return;
  const int64_t out = (KSIDE ? koff : qoff) + (int64_t)ri * sta_ld;
  if constexpr (MODE == MODE_FWD) {
    store_rows<T, D>((T*)p.o + out, acc0, 1.f / l, h);
    if (h == 0) p.lse[row] = (m + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;   // v_log_f32 is log2
  } else if constexpr (MODE == MODE_BWD_Q) {
    store_rows<T, D>((T*)p.dq + out, acc0, p.scale, h);
  } else {
    store_rows<T, D>((T*)p.dk + out, acc0, p.scale, h);
    store_rows<T, D>((T*)p.dv + out, acc1, 1.f, h);
  }
}

template <typename T, int D, int MODE, int MASK, int WS, bool TWO>
__global__ void __launch_bounds__(256, (min_workgroups<T, D, WS, TWO>)) attn_split(AttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  attn_run<T, D, MODE, MASK, WS, false, TWO>(p, smem, blockIdx.x, MASK != MASK_NONE && WS == 1 && min_workgroups<T, D, WS, TWO> == 2);
}

// dQ (workgroups [0, q_blocks)) and dK, dV (the others; mixed: tile by tile in turn) in one launch; ON_CU: workgroups on a CU
template <typename T, int D, int MASK, int WS, int ON_CU>
__global__ void __launch_bounds__(256, ON_CU) attn_split_bwd(AttnParams p, int q_blocks, bool mixed) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr bool joins = MASK != MASK_NONE && WS == 1 && ON_CU == 2;   // workgroups of a masked launch that share a CU
  int id = blockIdx.x;
  if (first_of_two(q_blocks, (int)gridDim.x - q_blocks, mixed, joins, id)) attn_run<T, D, MODE_BWD_Q, MASK, WS, false>(p, smem, id, joins && !mixed);
  else attn_run<T, D, MODE_BWD_K, MASK, WS, true>(p, smem, id, joins && !mixed);
}

template <typename T, int D, int MODE, int WS, bool TWO = false>
constexpr int lds_bytes() {
  constexpr bool KSIDE = MODE == MODE_BWD_K;
  constexpr int stages = n_buffers<WS, TWO> * WS * (Stager<T, D, 2, true, 0>::BYTES + (KSIDE ? 2 * TS * 4 : 0));
  constexpr int xch = WS > 1 ? (4 / WS) * (WS - 1) * ((KSIDE ? 2 : 1) * D / 32 * 16 + 2) * 64 * 4 : 0;
  return stages > xch ? stages : xch;
}

template <int WS>
unsigned blocks(int rows, int batch) { return grid_blocks((rows + 128 / WS - 1) / (128 / WS), batch); }

template <typename T, int D, int MODE, int MASK, int WS, bool TWO = false>
hipError_t launch_ws(const AttnParams& p, hipStream_t s) {
  constexpr int smem = lds_bytes<T, D, MODE, WS, TWO>();
  static_assert(smem <= 160 * 1024, "stages and exchange buffer have to fit the LDS");
  const hipError_t e = allow_dynamic_lds<attn_split<T, D, MODE, MASK, WS, TWO>>(smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((attn_split<T, D, MODE, MASK, WS, TWO>), dim3(blocks<WS>(MODE == MODE_BWD_K ? p.n_k : p.n_q, p.batch)), dim3(256), smem, s, p);
  return hipGetLastError();
}

template <typename T, int D, int MASK, int WS, int ON_CU = min_workgroups<T, D, WS, false>>
hipError_t launch_bwd_ws(const AttnParams& p, hipStream_t s, bool mixed = false) {
  constexpr int lq = lds_bytes<T, D, MODE_BWD_Q, WS>(), lk = lds_bytes<T, D, MODE_BWD_K, WS>(), smem = lq > lk ? lq : lk;
  static_assert(smem <= 160 * 1024, "stages and exchange buffer have to fit the LDS");
  const hipError_t e = allow_dynamic_lds<attn_split_bwd<T, D, MASK, WS, ON_CU>>(smem);
  if (e != hipSuccess) return e;
  const unsigned gq = blocks<WS>(p.n_q, p.batch), gk = blocks<WS>(p.n_k, p.batch);
  hipLaunchKernelGGL((attn_split_bwd<T, D, MASK, WS, ON_CU>), dim3(gq + gk), dim3(256), smem, s, p, (int)gq, mixed);
  return hipGetLastError();
}

// As in fhog_split.hip: four waves on 128 rows when that fills the GPU, two or four on the same 32 rows when it does not.
template <typename T, int D, int MASK>
hipError_t launch_fwd(const AttnParams& p, hipStream_t s) {
  const int64_t groups = (int64_t)(p.n_q + 127) / 128 * p.batch;
  if constexpr (lds_bytes<T, D, MODE_FWD, 4>() <= 160 * 1024) {
    if (groups < 64 && p.n_k > 2 * TS) return launch_ws<T, D, MODE_FWD, MASK, 4>(p, s);
  }
  if (groups < 128 && p.n_k > TS) return launch_ws<T, D, MODE_FWD, MASK, 2>(p, s);
  if constexpr (is_raw<T, D>) {
    if (rules::two_forwards_on_a_cu(groups, MASK != MASK_NONE)) return launch_ws<T, D, MODE_FWD, MASK, 1, true>(p, s);
  }
  return launch_ws<T, D, MODE_FWD, MASK, 1>(p, s);
}

template <typename T, int D, int MODE, int MASK>
hipError_t launch_side(const AttnParams& p, int waves, hipStream_t s) {
  if constexpr (lds_bytes<T, D, MODE, 4>() <= 160 * 1024) {
    if (waves == 4) return launch_ws<T, D, MODE, MASK, 4>(p, s);
  }
  return waves >= 2 ? launch_ws<T, D, MODE, MASK, 2>(p, s) : launch_ws<T, D, MODE, MASK, 1>(p, s);
}

// dQ and dK, dV side by side fill CUs for each other, as passes 3 and 4 do in fhog_split.hip, and the rule for waves on the same rows is of
// the same kind. The price is the row sums d, which the sweep for dK, dV then takes once per key block: nothing at d = 32 where the shared launch
// leaves CUs idle, up to a fifth where it does not or the key side is the longer one; 3 to 9 % on fp32 tensors of d = 64 and 128, whose launches of full rounds (256 workgroups each) go one after the other (split_bwd_waves). First backward,
// us, two launches (the rule before) -> one launch with four | two | one waves on the same rows:
//   bf16 d = 32   2 x 256 11.7 -> 7.9 | 9.8 | 12; causal 16 x 1024 56 -> 28 | 34 | 38, 64 x 1024 59 -> 81 | 57 | 49; no mask 16 x 1024 53 -> 37 | 35 | 37
//   fp32 d = 64   2 x 256 27 -> 16 | 21 | 31; causal 16 x 1024 181 -> 99 | 83 | 106, 32 x 1024 182 -> 192 | 135 | 122; no mask 48 x 1024
//                 309 -> - | 345 | 283, 64 x 1024 338 -> - | 459 | 362
//   fp32 d = 128  2 x 256 66 -> - | 46 | 59; causal 16 x 1024 325 -> - | 188 | 217, 64 x 1024 408 -> - | 620 | 428; no mask 64 x 1024 609 -> - | 989 | 631
template <typename T, int D, int MASK>
hipError_t launch_bwd(const AttnParams& p, hipStream_t s) {
  const int waves = rules::split_bwd_waves(p, sizeof(T));
  if (waves == 0) {
    const int64_t g_q = (int64_t)(p.n_q + 127) / 128 * p.batch, g_k = (int64_t)(p.n_k + 127) / 128 * p.batch;
    const hipError_t e = launch_side<T, D, MODE_BWD_Q, MASK>(p, rules::waves_of_side(g_q, p.n_k), s);
    return e != hipSuccess ? e : launch_side<T, D, MODE_BWD_K, MASK>(p, rules::waves_of_side(g_k, p.n_q), s);
  }
  if constexpr (lds_bytes<T, D, MODE_BWD_K, 4>() <= 160 * 1024) {
    if (waves == 4) return launch_bwd_ws<T, D, MASK, 4>(p, s);
  }
  if (waves >= 2) return launch_bwd_ws<T, D, MASK, 2>(p, s);
  if constexpr (sizeof(T) == 4 && D == 64 && MASK != MASK_NONE) {
    const rules::Company company = rules::bwd_company(p);
    return company == rules::Company::none ? launch_bwd_ws<T, D, MASK, 1, 1>(p, s) : launch_bwd_ws<T, D, MASK, 1>(p, s, company == rules::Company::in_turn);
  }
  if constexpr (sizeof(T) == 4 && D == 32 && MASK == MASK_NONE) {
    if (rules::bwd_company(p) == rules::Company::three) return launch_bwd_ws<T, D, MASK, 1, 3>(p, s);
  }
  return launch_bwd_ws<T, D, MASK, 1>(p, s, rules::split_in_turn(p, blocks<1>(p.n_q, p.batch), blocks<1>(p.n_k, p.batch)));
}

template <typename T, int D>
hipError_t launch_td(const AttnParams& p, bool backward, hipStream_t s) {
  if (backward) return p.causal ? launch_bwd<T, D, MASK_BAND>(p, s) : launch_bwd<T, D, MASK_NONE>(p, s);
  return p.causal ? launch_fwd<T, D, MASK_BAND>(p, s) : launch_fwd<T, D, MASK_NONE>(p, s);
}

}  // namespace

// dtype: FHOG_DTYPE_*. fp32 tensors of every head dim, 16-bit tensors of d = 32.
hipError_t launch_attn_split(const AttnParams& p, int dtype, bool backward, hipStream_t s) {
  if (dtype == FHOG_DTYPE_FP32) {
    switch (p.d) {
      case 32: return launch_td<float, 32>(p, backward, s);
      case 64: return launch_td<float, 64>(p, backward, s);
      case 128: return launch_td<float, 128>(p, backward, s);
      default: return hipErrorInvalidValue;
    }
  }
  if (p.d != 32) return hipErrorInvalidValue;
  return dtype == FHOG_DTYPE_FP16 ? launch_td<_Float16, 32>(p, backward, s) : launch_td<__bf16, 32>(p, backward, s);
}

}  // namespace fhog
