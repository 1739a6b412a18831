// Split-product kernels of the attention double-backward: products of fp32 accuracy on the 16-bit matrix instructions
// (fhog_split_util.h). They serve fp32 tensors and d = 32, and 16-bit tensors for which this family is asked for;
// fp32-accurate arithmetic throughout, no atomics, nothing of shape (N_Q, N_K) leaves the chip.
//
// One kernel template for the sweeps, with the arithmetic of the single-role 16-bit kernels (fhog_bf16.hip): a workgroup of
// 4 wave64 owns 32 stationary rows per wave (queries in passes 1-3 and 5, keys in pass 4) and keeps their operands in
// registers as bf16 terms; the other side streams through LDS in 32-row tiles, fetched into registers one step ahead,
// split into terms once per workgroup and read by all four waves. First-level products have the streamed rows as M and
// the stationary rows as N, so a lane owns ONE stationary row and its registers run over the streamed rows; split into
// terms, such a tile is as it stands the B operand of the second-level products, whose A operand is a transposing read of
// the staged tile in the same row order. Small launches (WS = 2 or 4) put WS waves on the same 32 rows instead: each takes
// every WS-th streamed tile and the partial results are added through LDS in a fixed order. Passes 3 and 4 share a launch (launch_grads).
//
// What bounds it: fp32 tensors the matrix pipe (216 MFMAs of 32 cycles per 32 x 32 block in pass 3 at d = 64, against 288 of
// 64 cycles as v_mfma_f32_32x32x2_f32), 16-bit tensors at d = 32 the VALU (34 MFMAs beside some 400
// VALU instructions, half of them the split of P, dS, dS' and ddP). A wave of fp32 tensors is alone on its SIMD (d >= 64), so whatever it does
// between two MFMAs the pipe waits for: LDS operands are read and numbers split behind the MFMAs of the step before (AHEAD, SecondLevel). Cycles of a
// step of pass 5 at d = 64 without a mask: 120 MFMAs 3936; all products 4260; with the next tile split and written behind them 5370, elementwise
// arithmetic 810, barrier 360 (splitting by itself: 1140 and 370 of requests more). Double-backward, us, without -> so: fp32 causal
// 32 x 2048 d = 128 pass 5 629 -> 561, passes 3 and 4 2021 -> 1978; d = 64 941 -> 920; no mask 40 x 1024, d = 64 704 -> 677; two workgroups of pass 5 on a
// CU (d = 64, numbers split again for every tile): 226 -> 319.
// Some do not quite fit the register file and keep bytes of a lane in scratch memory (spilled VGPRs as the compiler counts them, one that is spilled twice
// as two): fp32 tensors in passes 3 and 4 at d = 128 312 without a mask and 264 with one (110, 103), at d = 64 in the launch with two waves on the
// same rows beside four 160 and 208 (45, 51), with one wave at d = 32 24 and 40 (6, 11); 16-bit tensors at d = 128 up to 212 (52).
// Whole chain, us, against kernels on v_mfma_f32_32x32x2_f32 with the same tiling (same card):
//   bf16 causal 64 x 1024, d = 32: 734 -> 122     fp32 causal 64 x 1024, d = 32: 672 -> 272
//   fp32 causal 32 x 2048, d = 64: 2101 -> 919    fp32 64 x 2048, d = 64: 7521 -> 3453
//   fp32 causal 32 x 2048, d = 128: 3833 -> 2190
// and no result is less accurate: against fp64, fp32 outputs are off by 3e-7 to 1.2e-6 (2-norm) either way.
//
// Math per tile pair (fhog/triton_bwdbwd.py:194-202, 229-243, 266-288, 485-507), with u = dP - d, w = ddS - dd:
//   S = scale Q K^T, P = exp(S - L), dP = dO V^T, ddS = scale (ddQ K^T + Q ddK^T), E' = dO ddV^T - dd d - b
//   dS = scale P u, ddP = P w, dS' = scale (P E' + ddP u)
#include <type_traits>

#include "fhog_rules.h"
#include "fhog_split_util.h"

namespace fhog {
using namespace splitk;
namespace {

// Stages of the ring: two where they fit (a wave split stages WS tiles at a time instead).
template <typename T, int D, int WS>
constexpr int n_buffers(int stage) { return WS == 1 && !is_raw<T, D> && 2 * stage <= 160 * 1024 ? 2 : 1; }

// A statistics sweep whose four waves share their rows: each streamed tile has one reader, and its rows as they lie in memory
// are the A operand of the first level, which is all these sweeps have. The wave loads them two k-steps ahead straight into
// registers: no staging through LDS, no barriers, and no LDS limit on the split (fp32: two tiles of four tensors at d = 64, one
// at 128). Pass 5, us, staged -> direct: fp32 2 x 256, d = 64 20.8 -> 14.1; fp32 causal 1 x 4096, d = 128 977 -> 240;
// fp32 causal 1 x 6000, d = 64 365 -> 169; bf16 1 x 8000, d = 32 66 -> 38; bf16 causal 2 x 512, d = 32 7.3 -> 6.0.
template <int PASS, int WS>
constexpr bool is_direct = WS == 4 && (PASS == 1 || PASS == 2 || PASS == 5);

// PASS 1: d, dd; 2: b; 3: dQ2, ddO; 4: dK2, dV2 (K-tiled); 5: d, dd, b.
// pairs: as decode_block takes it
template <typename T, int D, int PASS, int MASK, int WS>
__device__ __forceinline__ void split_run(const Params& p, char* smem, int id, bool pairs) {
  constexpr bool KSIDE = PASS == 4, STATS = PASS == 1 || PASS == 2 || PASS == 5;
  constexpr int NT = PASS == 1 ? 2 : (KSIDE ? 3 : 4);      // streamed tensors: K, ddK, V, ddV | Q, ddQ, dO
  constexpr int NR = PASS == 1 ? 2 : (KSIDE ? 4 : 3);      // stationary tensors: Q, ddQ, dO | K, ddK, V, ddV
  constexpr int KK = D / 16, NC = D / 32, NF = Terms<T>::NF;
  // An infinity in K, ddK, Q or ddQ makes a NaN of dd and, with it, of whole rows; one in V, ddV or dO leaves other columns of
  // ddO or dV2 as they are. The statistics sweeps have sums over rows only.
  using Stage = Stager<T, D, NT, !STATS, STATS ? NT : 2>;
  constexpr int TENSOR = Stage::PLANES * Stage::TILE;
  constexpr int STAT = KSIDE ? 4 * TS * 4 : 0;             // L log2(e), -d, dd, -(dd d + b) of the 32 staged queries
  constexpr int STAGE = Stage::BYTES + STAT;
  // fp32, d = 128: the terms of three or four stationary tensors are 288 or 384 registers, so the wave keeps the fp32 numbers
  // (the last tensor of passes 3 and 4, dO or ddV, in LDS) and splits them again for every tile, one k-step at a time, in the statistics sweeps behind the
  // MFMAs of the one before: 28 VALU instructions per tensor and k-step beside 30 MFMAs.
  constexpr bool RAW = is_raw<T, D>;
  constexpr bool LAST_IN_LDS = RAW && !STATS;
  constexpr int NREG = LAST_IN_LDS ? NR - 1 : NR;
  constexpr bool DIRECT = is_direct<PASS, WS>;
  // A wave is alone on its SIMD: what it waits for is put behind its own MFMAs. At d = 128 the first level of passes 3 and 4 has no registers for that.
  constexpr bool AHEAD2 = sizeof(T) == 4 && D >= 64 && !DIRECT && PASS != 1, AHEAD = AHEAD2 && !LAST_IN_LDS;
  constexpr int NBUF = n_buffers<T, D, WS>(STAGE);
  constexpr int nw = 4 / WS, ROWS = 32 * nw;

  constexpr bool INTERLEAVED = AHEAD && STATS && WS == 1 && NBUF == 2;   // the next tile is split and written to LDS behind the MFMAs of this one

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wv / WS, ws = wv % WS;   // row group of the wave, and which of the streamed tiles of a step it takes
  const int n = lane & 31, h = lane >> 5;
  const int n_sta = KSIDE ? p.n_k : p.n_q, n_str = KSIDE ? p.n_q : p.n_k;
  int bh, tile;
  if (!decode_block<MASK>((n_sta + ROWS - 1) / ROWS, p.batch, !KSIDE && MASK != MASK_NONE, KSIDE ? p.tile_major_k : p.tile_major, bh, tile, pairs, id)) return;
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb;
  const int64_t sta_ld = KSIDE ? p.stride_kn : p.stride_qn, str_ld = KSIDE ? p.stride_qn : p.stride_kn;
  const int r0 = tile * ROWS, rw = r0 + 32 * group, ri = rw + n;
  const int rr = min(ri, n_sta - 1);         // rows past the end compute on a copy of the last row and store nothing
  const T* src[NT];
  if constexpr (KSIDE) {
    src[0] = (const T*)p.q + qoff, src[1] = (const T*)p.ddq + qoff, src[2] = (const T*)p.dO + qoff;
  } else {
    src[0] = (const T*)p.k + koff, src[1] = (const T*)p.ddk + koff;
    if constexpr (NT == 4) src[2] = (const T*)p.v + koff, src[3] = (const T*)p.ddv + koff;
  }

  typename std::conditional<KSIDE, StreamQueries<MASK>, StreamKeys<MASK>>::type geo(p.mask_off, p.window, n_str);
  int t_begin, t_end;
  geo.tile_range(r0, ROWS, t_begin, t_end);

  const int64_t srow = (int64_t)bh * p.n_q;
  Stage st[WS];
  float stat_reg[WS] = {}, stat_d[WS] = {}, stat_dd[WS] = {};
  // pass 4: threads t and t + 128 carry statistic t / 32 of staged query t % 32. All of them without a branch, or 128 that load what they need, us: fp32
  // causal 64 x 1024, d = 32 271 | 276; no mask bf16 d = 32 2 x 256 11.9 | 13.4, 8 x 512 18.0 | 20.0, 16 x 4096 705 | 702; others within 0.5 %.
  const int which = (tid >> 5) & 3;
  const float* const stat_src = which == 0 ? p.lse : which == 1 ? p.ws_d : which == 2 ? p.ws_dd : p.ws_b;
  const auto fetch = [&](int t) {
#pragma unroll
    for (int g = 0; g < WS; g++) {
      const int row0 = (t + g) * TS;
      st[g].fetch(src, str_ld, min(row0, n_str - 1), n_str, tid);   // a tile past the end is never computed on
      if constexpr (KSIDE) {
        const int64_t q = srow + min(row0 + (tid & 31), p.n_q - 1);
        stat_reg[g] = stat_src[q], stat_d[g] = p.ws_d[q], stat_dd[g] = p.ws_dd[q];
      }
    }
  };
  const auto publish = [&](int buf) {
#pragma unroll
    for (int g = 0; g < WS; g++) {
      char* stage = smem + (buf * WS + g) * STAGE;
      st[g].publish(stage, tid);
      if constexpr (KSIDE) {
        reinterpret_cast<float*>(stage + Stage::BYTES)[tid & 127] =
            which == 0 ? stat_reg[g] * kLog2e : which == 1 ? -stat_reg[g] : which == 2 ? stat_reg[g] : -__builtin_fmaf(stat_dd[g], stat_d[g], stat_reg[g]);
      }
    }
  };
  if (!DIRECT && t_begin < t_end) fetch(t_begin);

  const T* const sta[4] = {KSIDE ? (const T*)p.k + koff : (const T*)p.q + qoff, KSIDE ? (const T*)p.ddk + koff : (const T*)p.ddq + qoff,
                           KSIDE ? (const T*)p.v + koff : (const T*)p.dO + qoff, (const T*)p.ddv + koff};
  Resident<T, D> res[NREG];
#pragma unroll
  for (int x = 0; x < NREG; x++) res[x].load(sta[x] + (int64_t)rr * sta_ld, h);
  // the last tensor of the wave's rows, 16 bytes of a lane beside those of the next one
  f32x4_t* const last = reinterpret_cast<f32x4_t*>(smem + NBUF * WS * STAGE) + wv * (KK * 2 * 64) + lane;
  if constexpr (LAST_IN_LDS) {
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
      const Chunk<T> c = load_chunk<T>(sta[NR - 1] + (int64_t)rr * sta_ld + 16 * kk + 8 * h);
      last[(2 * kk) * 64] = __builtin_bit_cast(f32x4_t, c.v[0]);
      last[(2 * kk + 1) * 64] = __builtin_bit_cast(f32x4_t, c.v[sizeof(T) / 2 - 1]);
    }
  }
  const int64_t row = srow + rr;   // Q-tiled passes
  float l_log2 = 0.f, dsum = 0.f, dd = 0.f, b = 0.f;
  if constexpr (!KSIDE) {
    l_log2 = p.lse[row] * kLog2e;
    if constexpr (PASS == 1 || PASS == 5) {
      // d_i = sum_c O_ic dO_ic (fhog/triton_bwdbwd.py:580): each lane takes half of its query's row
#pragma unroll
      for (int kk = 0; kk < KK; kk++) {
        const Chunk<T> o = load_chunk<T>((const T*)p.o + qoff + (int64_t)rr * sta_ld + 16 * kk + 8 * h);
        const Chunk<T> g = load_chunk<T>((const T*)p.dO + qoff + (int64_t)rr * sta_ld + 16 * kk + 8 * h);
#pragma unroll
        for (int e = 0; e < 8; e++) dsum = __builtin_fmaf(chunk_elem(o, e), chunk_elem(g, e), dsum);
      }
      dsum += __shfl_xor(dsum, 32);
      if (h == 0 && ri < p.n_q && ws == 0) p.ws_d[row] = dsum;
    } else {
      dsum = p.ws_d[row], dd = p.ws_dd[row];
      if constexpr (PASS == 3) b = p.ws_b[row];
    }
  }
  const float kc = __builtin_fmaf(dd, dsum, b);
  const float c_scale_log2 = p.scale * kLog2e;

  // AHEAD: the other offsets follow from these by an exclusive or; kept in registers, they would be spilled
  int aoff0 = tile_off<D>(n, h), tr0 = tr_lane_off_acc<D>(0, 0, lane), tr1 = tr_lane_off_acc<D>(0, 1, lane);
  int aoff[KK], troff[NC][2];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) aoff[kk] = tile_off<D>(n, 2 * kk + h);
#pragma unroll
  for (int cb = 0; cb < NC; cb++) troff[cb][0] = tr_lane_off_acc<D>(cb, 0, lane), troff[cb][1] = tr_lane_off_acc<D>(cb, 1, lane);

  f32x16_t acc0[NC], acc1[NC];     // dQ2, ddO | dK2, dV2: lane = stationary row, registers = columns
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc0[cb] = f32x16_t{0}, acc1[cb] = f32x16_t{0};
  float red[5] = {};               // statistics: b-like sum; fused sweep: dd, sum P u ddS, sum P u, sum P

  Chunk<T> ahead[2][NT];           // DIRECT: the next two k-steps of the lane's streamed row
  const auto load_step = [&](int t, int kk) {
    const int64_t off = (int64_t)min(t * TS + n, n_str - 1) * str_ld + 16 * kk + 8 * h;
#pragma unroll
    for (int x = 0; x < NT; x++) ahead[kk & 1][x] = load_chunk<T>(src[x] + off);
  };

  // AHEAD: the first level of one tile for a lone wave on its SIMD. What a group of MFMAs takes from LDS is read, and the terms that it
  // takes of a stationary row are split (RAW), behind the MFMAs of the group before; the fences hold that order. Two chains
  // of products take turns where a group has two.
  const auto first_level = [&](const char* stage, int s0, f32x16_t& s, f32x16_t& dds, f32x16_t& dp, f32x16_t& e, auto behind) {
    constexpr TermPairs<NF, NF> kPairs{};
    bf16x8_t a[NT][NF];
    Splitting<NF> terms[NR];   // RAW
    const auto read = [&](int x, int kk) { read_terms<T, Stage::TILE>(stage + x * TENSOR, aoff0 ^ (32 * kk), a[x]); };
    // what is due behind MFMA `slot` of `slots` of the terms of k-step kk of stationary tensor y
    const auto split = [&](int y, int kk, int slot, int slots) {
      if constexpr (RAW) {
        const Chunk<T>& c = res[y].r[kk];
        terms[y].at(slot, slots, [&](int i, float& lo, float& hi) {
          lo = chunk_elem(c, 2 * i), hi = chunk_elem(c, 2 * i + 1);
          asm("" : "+v"(lo), "+v"(hi) : "s"(s0));   // here, tile after tile: hoisted out of the sweep, the terms would be spilled
        });
      }
    };
    const auto sta_term = [&](int y, int kk, int q) {
      if constexpr (RAW) return terms[y].term(q);
      else return res[y].r[kk][q];
    };
    constexpr int P = kPairs.n;
    read(0, 0), read(1, 0);
    split(0, 0, 0, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
#pragma unroll
      for (int i = 0; i < P; i++) {
        s = mfma<false>(a[0][kPairs.a[i]], sta_term(0, kk, kPairs.b[i]), s);         // K Q^T | Q K^T
        split(1, kk, 2 * i, 2 * P);
        behind(5 * P * kk + 2 * i, 5 * P * KK);
        __builtin_amdgcn_sched_barrier(0);
        dds = mfma<false>(a[1][kPairs.a[i]], sta_term(0, kk, kPairs.b[i]), dds);     // ddK Q^T | ddQ K^T
        if (i == 0) read(2, kk);
        if (!KSIDE && i == 1) read(NT - 1, kk);
        split(1, kk, 2 * i + 1, 2 * P);
        behind(5 * P * kk + 2 * i + 1, 5 * P * KK);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < P; i++) {
        dds = mfma<false>(a[0][kPairs.a[i]], sta_term(1, kk, kPairs.b[i]), dds);     // + K ddQ^T | Q ddK^T
        split(NR - 1, kk, i, P);
        behind(5 * P * kk + 2 * P + i, 5 * P * KK);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < P; i++) {
        dp = mfma<false>(a[2][kPairs.a[i]], sta_term(2, kk, kPairs.b[i]), dp);       // V dO^T | dO V^T
        if (kk + 1 < KK) {
          if (i == 0) read(0, kk + 1), read(1, kk + 1);
          split(0, kk + 1, 2 * i, 2 * P);
        }
        behind(5 * P * kk + 3 * P + 2 * i, 5 * P * KK);
        __builtin_amdgcn_sched_barrier(0);
        e = mfma<false>(a[NT - 1][kPairs.a[i]], sta_term(NR - 1, kk, kPairs.b[i]), e);   // ddV dO^T | dO ddV^T
        if (kk + 1 < KK) split(0, kk + 1, 2 * i + 1, 2 * P);
        behind(5 * P * kk + 3 * P + 2 * i + 1, 5 * P * KK);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // holds the products in front of the branches that follow: the compiler sinks a chain of MFMAs to the block that uses its sum
    asm volatile("" : "+v"(s), "+v"(dds), "+v"(dp), "+v"(e));
  };

  // prefetch: what requests the next tile; called where the registers it lands in are free
  // behind(slot, slots): what is to be done behind MFMA `slot` of the first level (AHEAD)
  const auto block = [&](const char* stage, int s0, auto prefetch, auto behind) {
    const float* stat = reinterpret_cast<const float*>(stage + Stage::BYTES);
    f32x16_t s = {0}, dds = {0}, dp = {0}, e = {0};
    // u = dP - d and E' = E - (dd d + b) come straight from accumulators that start at the row constants
    if constexpr (KSIDE) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x4_t md4 = *reinterpret_cast<const f32x4_t*>(stat + 1 * TS + 8 * g + 4 * h);
        const f32x4_t mk4 = *reinterpret_cast<const f32x4_t*>(stat + 3 * TS + 8 * g + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; i++) dp[4 * g + i] = md4[i], e[4 * g + i] = mk4[i];
      }
    } else if constexpr (PASS != 1) {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        dp[r] = -dsum;
        if (PASS != 5) e[r] = -kc;
      }
    }
    if constexpr (AHEAD2) asm volatile("" : "+v"(tr0), "+v"(tr1));
    if constexpr (AHEAD) {
      asm volatile("" : "+v"(aoff0));
      first_level(stage, s0, s, dds, dp, e, behind);
    } else {
#pragma unroll
      for (int kk = 0; kk < KK; kk++) {
        bf16x8_t r0[NF], r1[NF], r2[NF], r3[NF], a[NF];
        res[0].terms(kk, r0), res[1].terms(kk, r1);
        const auto last_terms = [&](bf16x8_t (&out)[NF]) {
          if constexpr (LAST_IN_LDS) {
            Chunk<T> c;
            c.v[0] = __builtin_bit_cast(u32x4_t, last[(2 * kk) * 64]), c.v[sizeof(T) / 2 - 1] = __builtin_bit_cast(u32x4_t, last[(2 * kk + 1) * 64]);
            chunk_terms<T, true, false>(c, out);
          } else {
            res[NREG - 1].terms(kk, out);
          }
        };
        if constexpr (KSIDE) res[2].terms(kk, r2), last_terms(r3);
        else if constexpr (PASS != 1) last_terms(r2);
        const auto streamed = [&](int x) {
          if constexpr (DIRECT) chunk_terms<T, true, false>(ahead[kk & 1][x], a);
          else read_terms<T, Stage::TILE>(stage + x * TENSOR, aoff[kk], a);
        };
        streamed(0);
        s = mma1<T>(s, a, r0);                                  // K Q^T | Q K^T
        dds = mma1<T>(dds, a, r1);                              // K ddQ^T | Q ddK^T
        if constexpr (PASS != 1) {
          streamed(2);
          dp = mma1<T>(dp, a, r2);                              // V dO^T | dO V^T
          if constexpr (KSIDE) e = mma1<T>(e, a, r3);           // dO ddV^T
        }
        streamed(1);
        dds = mma1<T>(dds, a, r0);                              // + ddK Q^T | ddQ K^T
        if constexpr (PASS != 1 && !KSIDE) {
          streamed(NT - 1);
          e = mma1<T>(e, a, r2);                                // ddV dO^T
        }
        if constexpr (DIRECT) load_step(s0 / TS + (kk + 2 < KK ? 0 : WS), (kk + 2) % KK);   // past the last tile: its last row again
        if constexpr (RAW || DIRECT) __builtin_amdgcn_sched_barrier(0);
      }
    }
    f32x16_t pv;
#pragma unroll
    for (int g = 0; g < 4; g++) {
      f32x4_t l4 = {l_log2, l_log2, l_log2, l_log2};
      if constexpr (KSIDE) l4 = *reinterpret_cast<const f32x4_t*>(stat + 8 * g + 4 * h);
#pragma unroll
      for (int i = 0; i < 4; i++) pv[4 * g + i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * g + i], c_scale_log2, -l4[i]));
    }
    if (RAW && MASK != MASK_NONE) {
      int lo, hi;
      geo.limits(s0, ri, h, lo, hi);
#pragma unroll
      for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
    } else if (geo.partial(s0, rw)) {   // wave-uniform: the block holds hidden pairs (mask edge or tensor end)
      int lo, hi;
      geo.limits(s0, ri, h, lo, hi);
      keep_branch();
#pragma unroll
      for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
    }
    if constexpr (PASS == 1) {
#pragma unroll
      for (int r = 0; r < 16; r++) red[1] = __builtin_fmaf(pv[r], dds[r], red[1]);
    } else if constexpr (PASS == 2) {
#pragma unroll
      for (int r = 0; r < 16; r++) red[0] = __builtin_fmaf(pv[r], __builtin_fmaf(__builtin_fmaf(dds[r], p.scale, -dd), dp[r], e[r]), red[0]);
    } else if constexpr (PASS == 5) {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float v = pv[r] * dp[r];
        red[0] = __builtin_fmaf(pv[r], e[r], red[0]);
        red[1] = __builtin_fmaf(pv[r], dds[r], red[1]);
        red[2] = __builtin_fmaf(v, dds[r], red[2]);
        red[3] += v;
        red[4] += pv[r];
      }
    } else if constexpr (AHEAD2) {
      f32x4_t dd4[4];
#pragma unroll
      for (int g = 0; g < 4; g++) {
        if constexpr (KSIDE) dd4[g] = *reinterpret_cast<const f32x4_t*>(stat + 2 * TS + 8 * g + 4 * h);
      }
      const auto elementwise = [&](int r) {
        if (r < 0 || r >= 16) return;
        dds[r] = pv[r] * __builtin_fmaf(dds[r], p.scale, KSIDE ? -dd4[r / 4][r % 4] : -dd);   // ddP = P w
        if (!KSIDE) s[r] = pv[r] * dp[r];                                                      // dS = P u (scale applied to the accumulators at the end)
        e[r] = __builtin_fmaf(pv[r], e[r], dds[r] * dp[r]);                                    // dS' = P E' + ddP u
      };
      SecondLevel<T, D> second{tr0, tr1};
      if constexpr (!KSIDE) {
        second.start(stage + (NT - 1) * TENSOR, pv);
        second.template run<true>(acc1, stage + (NT - 1) * TENSOR, pv, stage + TENSOR, s, elementwise);         // ddO += P ddV
        second.template run<true>(acc0, stage + TENSOR, s, stage + 2 * TENSOR, dds, [](int) {});                // dQ2 += dS ddK
      } else {
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = pv[r] * dp[r];
        second.start(stage + TENSOR, s);
        second.template run<true>(acc0, stage + TENSOR, s, stage + 2 * TENSOR, dds, elementwise);               // dK2 += dS^T ddQ
      }
      second.template run<true>(acc1, stage + 2 * TENSOR, dds, stage, e, [](int) {});                           // ddO += ddP V | dV2 += ddP^T dO
      prefetch();
      second.template run<false>(acc0, stage, e, stage, e, [](int) {});                                         // dQ2 += dS' K | dK2 += dS'^T Q
    } else {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        f32x4_t dd4 = {dd, dd, dd, dd};
        if constexpr (KSIDE) dd4 = *reinterpret_cast<const f32x4_t*>(stat + 2 * TS + 8 * g + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int r = 4 * g + i;
          dds[r] = pv[r] * __builtin_fmaf(dds[r], p.scale, -dd4[i]);   // ddP = P w
          s[r] = pv[r] * dp[r];                                         // dS = P u (scale applied to the accumulators at the end)
          e[r] = __builtin_fmaf(pv[r], e[r], dds[r] * dp[r]);           // dS' = P E' + ddP u
        }
      }
      if constexpr (!KSIDE) second_level<T, D>(acc1, stage + (NT - 1) * TENSOR, troff, pv);   // ddO += P ddV
      second_level<T, D>(acc0, stage + 1 * TENSOR, troff, s);           // dQ2 += dS ddK | dK2 += dS^T ddQ
      second_level<T, D>(acc1, stage + 2 * TENSOR, troff, dds);         // ddO += ddP V | dV2 += ddP^T dO
      second_level<T, D>(acc0, stage, troff, e);                        // dQ2 += dS' K | dK2 += dS'^T Q
    }
  };

  constexpr bool LATE = RAW && !STATS;   // the next tile is requested towards the end of a step: no registers for it before
  if constexpr (DIRECT) {
    // the range of 32 rows holds no tile that is dead to the wave
    if (t_begin + ws < t_end) load_step(t_begin + ws, 0), load_step(t_begin + ws, 1);
    for (int t = t_begin + ws; t < t_end; t += WS) block(smem, t * TS, [] {}, [](int, int) {});
  }
  if (!DIRECT && t_begin < t_end) publish(0);
  if (INTERLEAVED && t_begin < t_end) fetch(t_begin + 1);
  if (!DIRECT) __syncthreads();
  // Without a mask only waves whose rows all lie past the end of the tensor see nothing. At d = 32 they have a loop of their own, for the test in the loop
  // costs every length: double-backward, us, neither | the test | two loops: bf16 16 x 4096 701 | 710 | 697, 64 x 1024 183 | 185 | 183, fp32 16 x 1000 159 |
  // 163 | 160, 16 x 4096 1835 | 1836 | 1822, 128 x 300 124 | 119 | 118. At d = 64 the test is the faster (fp32 16 x 2048 878 | 888), and in passes 3 and 4
  // of fp32 tensors at d = 128, which spill less with its branch, whichever mask. Double-backward, us, every tile computed | the test: no mask 32 x 2048 4131 |
  // 3986, 40 x 300 199 | 193, 2000 | 900 rows 1524 | 1459; causal 32 x 2048 2262 | 2156, 48 x 1537 2244 | 2130; window 700 16 x 1000 x 3000 569 | 541.
  constexpr bool NO_TEST = MASK == MASK_NONE && D == 32;
  const auto sweep = [&](auto has_rows) {
    const auto works = [&](int s0) { return NO_TEST ? decltype(has_rows)::value : !geo.dead(s0, geo.first_row(rw, n_sta)); };
    for (int t = t_begin; !DIRECT && t < t_end; t += WS) {
      const int buf = NBUF == 2 ? (t - t_begin) & 1 : 0;
      const int s0 = (t + ws) * TS;
      if constexpr (INTERLEAVED) {
        // The rows of the tile after this one came in during the step before; behind the last tile they are copies of the last row.
        char* const next = smem + (buf ^ 1) * STAGE;
        const int row0 = min(s0 + 2 * TS, n_str - 1);
        if (works(s0)) {
          block(smem + buf * STAGE, s0, [] {}, [&](int slot, int slots) {
            st[0].publish_at(next, tid, slot, slots, [&](int i) { st[0].fetch_chunk(i, src, str_ld, row0, n_str, tid); });
          });
        } else {
          publish(buf ^ 1);
          fetch(t + 2);
        }
        __syncthreads();
      } else {
        const bool more = t + WS < t_end;
        const auto next = [&]() {
          if (more) fetch(t + WS);
        };
        if (!LATE) next();
        if ((WS == 1 || t + ws < t_end) && works(s0)) {
          block(smem + (buf * WS + ws) * STAGE, s0, [&]() {
            if (LATE) {
              __builtin_amdgcn_sched_barrier(0);
              next();
              __builtin_amdgcn_sched_barrier(0);
            }
          }, [](int, int) {});
        } else if (LATE) {
          next();
        }
        if (NBUF == 1) __syncthreads();   // the tiles are no longer read
        if (more) publish(NBUF == 2 ? buf ^ 1 : 0);
        __syncthreads();
      }
    }
  };
  if (NO_TEST && rw >= n_sta) sweep(std::false_type{});
  else sweep(std::true_type{});

  if constexpr (WS > 1) {
    // the WS waves of a row group add their partial results in the order of ws; the wave with ws == 0 holds the sum
    constexpr int VALS = STATS ? 5 : 2 * NC * 16;
    float* const xch = reinterpret_cast<float*>(smem) + lane;
    const auto each = [&](auto f) {
      if constexpr (STATS) {
#pragma unroll
        for (int i = 0; i < 5; i++) f(red[i], i);
      } else {
#pragma unroll
        for (int cb = 0; cb < NC; cb++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            float x = acc0[cb][r], y = acc1[cb][r];
            f(x, cb * 16 + r), f(y, (NC + cb) * 16 + r);
            acc0[cb][r] = x, acc1[cb][r] = y;
          }
      }
    };
    if (ws > 0) each([&](float& x, int i) { xch[((group * (WS - 1) + ws - 1) * VALS + i) * 64] = x; });
    __syncthreads();
    if (ws > 0) return;
#pragma unroll
    for (int o = 1; o < WS; o++) each([&](float& x, int i) { x += xch[((group * (WS - 1) + o - 1) * VALS + i) * 64]; });
  }

  if constexpr (STATS) {
#pragma unroll
    for (int i = 0; i < 5; i++) red[i] += __shfl_xor(red[i], 32);
    if (h != 0 || ri >= p.n_q) return;
    if constexpr (PASS == 2) {
      p.ws_b[row] = red[0];
    } else {
      const float dd_i = red[1] * p.scale;
      p.ws_dd[row] = dd_i;
      if constexpr (PASS == 5)   // sum P (E + ddS u) - dd sum P dP
        p.ws_b[row] = __builtin_fmaf(-dd_i, __builtin_fmaf(dsum, red[4], red[3]), __builtin_fmaf(p.scale, red[2], red[0]));
    }
  } else {
    if (ri >= n_sta) return;
    const int64_t out = (KSIDE ? koff : qoff) + (int64_t)ri * sta_ld;
    store_rows<T, D>((T*)(KSIDE ? p.dk2 : p.dq2) + out, acc0, p.scale, h);
    store_rows<T, D>((T*)(KSIDE ? p.dv2 : p.ddo) + out, acc1, 1.f, h);
  }
}

template <int D, int WS>
constexpr int min_workgroups = D >= 64 || WS > 1 ? 1 : 2;

// workgroups of a masked launch that share a CU
template <int D, int MASK, int WS>
constexpr bool joins = MASK != MASK_NONE && D < 64 && WS == 1;

template <typename T, int D, int PASS, int MASK, int WS>
__global__ void __launch_bounds__(256, (min_workgroups<D, WS>)) split_sweep(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  split_run<T, D, PASS, MASK, WS>(p, smem, blockIdx.x, joins<D, MASK, WS>);
}

// Passes 3 (workgroups [0, q_blocks)) and 4 (the others; mixed: tile by tile in turn) in one launch: given the row statistics neither needs the other.
template <typename T, int D, int MASK, int WS3, int WS4>
__global__ void __launch_bounds__(256, (min_workgroups<D, (WS3 > WS4 ? WS3 : WS4)>)) split_grads(Params p, int q_blocks, bool mixed) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  int id = blockIdx.x;
  if (first_of_two(q_blocks, (int)gridDim.x - q_blocks, mixed, joins<D, MASK, WS3>, id)) split_run<T, D, 3, MASK, WS3>(p, smem, id, joins<D, MASK, WS3> && !mixed);
  else split_run<T, D, 4, MASK, WS4>(p, smem, id, joins<D, MASK, WS4> && !mixed);
}

template <typename T, int D, int PASS, int WS>
constexpr int lds_bytes() {
  constexpr bool KSIDE = PASS == 4, STATS = PASS == 1 || PASS == 2 || PASS == 5;
  constexpr int NT = PASS == 1 ? 2 : (KSIDE ? 3 : 4), nw = 4 / WS;
  constexpr int stage = Stager<T, D, NT, !STATS, 0>::BYTES + (KSIDE ? 4 * TS * 4 : 0);
  constexpr int stages = is_direct<PASS, WS> ? 0 : n_buffers<T, D, WS>(stage) * WS * stage + (is_raw<T, D> && !STATS ? 4 * TS * D * 4 : 0);
  constexpr int xch = WS > 1 ? nw * (WS - 1) * (STATS ? 5 : 2 * D / 32 * 16) * 64 * 4 : 0;
  return stages > xch ? stages : xch;
}

template <typename T, int D, int PASS, int MASK, int WS>
hipError_t launch_ws(const Params& p, hipStream_t s) {
  constexpr int smem = lds_bytes<T, D, PASS, WS>(), nw = 4 / WS;
  static_assert(smem <= 160 * 1024, "stages and exchange buffer have to fit the LDS");
  const hipError_t e = allow_dynamic_lds<split_sweep<T, D, PASS, MASK, WS>>(smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((split_sweep<T, D, PASS, MASK, WS>), dim3(grid_blocks((p.n_q + 32 * nw - 1) / (32 * nw), p.batch)), dim3(256), smem, s, p);
  return hipGetLastError();
}

// Four waves on 128 stationary rows share the streamed tiles and their splitting, the best shape whenever that fills the GPU
// (256 CUs). With fewer than 128 (64) such workgroups two (four) waves go on the same 32 rows, where the tiles of a step fit
// the LDS (four waves of a statistics sweep stage nothing): two fp32 heads of 256 tokens are 4 workgroups otherwise, each running its eight streamed tiles one after the other.
// A statistics sweep that stages nothing splits every tile into terms once per 32 rows instead of once per 128, but its workgroups
// are a quarter of the size: worth it beyond 64 workgroups where the staged form leaves CUs to the heaviest tiles of a causal
// triangle, or has one wave per row block. Statistics sweeps only; passes 3 and 4 are launch_grads' below. Pass 5, us, staged -> direct, at so many 128-row workgroups:
// Left as it is: triangles of 160 to 255 workgroups on fp32 tensors at d <= 64, where 15 x 2048 would gain (d = 64: 185 -> 151) what
// 60 x 500 would lose (the number of streamed tiles tells them apart), and windows and bottom-right masks beyond 128 (fp32
// d <= 64: 64), which were not measured.
//   triangle: fp32 d = 128 497 -> 130 (64), 502 -> 302 (240); bf16 d = 32 43.7 -> 24.7 (240), 60 x 500 14.0 -> 11.5 (240);
//             fp32 d = 64 184 -> 82 (128), but 60 x 500 52.2 -> 60.4 (240)
//   no mask:  fp32 d = 128 553 -> 435 (126); bf16 d = 32 43.0 -> 32.5 (126); fp32 d = 64 129 -> 137 (96)
template <typename T, int D, int PASS, int MASK>
hipError_t launch_sweep(const Params& p, hipStream_t s) {
  const int64_t groups = (int64_t)(p.n_q + 127) / 128 * p.batch;
  const bool triangle = MASK != MASK_NONE && p.mask_off == 0 && p.window >= p.n_k;
  constexpr bool splits_dear = sizeof(T) == 4 && D < 128;
  const int64_t line = triangle ? (splits_dear ? 160 : 256) : splits_dear ? 64 : 128;
  if (groups < line && p.n_k > 2 * TS) return launch_ws<T, D, PASS, MASK, 4>(p, s);
  if constexpr (lds_bytes<T, D, PASS, 2>() <= 160 * 1024) {
    if (groups < 128 && p.n_k > TS) return launch_ws<T, D, PASS, MASK, 2>(p, s);
  }
  return launch_ws<T, D, PASS, MASK, 1>(p, s);
}

template <int WS>
unsigned blocks(int rows, int batch) { return grid_blocks((rows + 128 / WS - 1) / (128 / WS), batch); }

// At most MOST waves on the same rows, as many as let either pass fit the LDS. sides: 1 pass 3, 2 pass 4, 3 both
template <typename T, int D, int MASK, int MOST>
hipError_t launch_grads_most(const Params& p, int sides, hipStream_t s) {
  constexpr int ws3 = MOST >= 4 && lds_bytes<T, D, 3, 4>() <= 160 * 1024 ? 4 : MOST >= 2 && lds_bytes<T, D, 3, 2>() <= 160 * 1024 ? 2 : 1;
  constexpr int ws4 = MOST >= 4 && lds_bytes<T, D, 4, 4>() <= 160 * 1024 ? 4 : MOST >= 2 && lds_bytes<T, D, 4, 2>() <= 160 * 1024 ? 2 : 1;
  constexpr int l3 = lds_bytes<T, D, 3, ws3>(), l4 = lds_bytes<T, D, 4, ws4>(), smem = l3 > l4 ? l3 : l4;
  static_assert(smem <= 160 * 1024, "stages and exchange buffer have to fit the LDS");
  const hipError_t e = allow_dynamic_lds<split_grads<T, D, MASK, ws3, ws4>>(smem);
  if (e != hipSuccess) return e;
  const unsigned gq = sides & 1 ? blocks<ws3>(p.n_q, p.batch) : 0, gk = sides & 2 ? blocks<ws4>(p.n_k, p.batch) : 0;
  hipLaunchKernelGGL((split_grads<T, D, MASK, ws3, ws4>), dim3(gq + gk), dim3(256), smem, s, p, (int)gq, ws3 == 1 && ws4 == 1 && rules::split_in_turn(p, gq, gk));
  return hipGetLastError();
}

template <typename T, int D, int MASK>
hipError_t launch_grads_side(const Params& p, int sides, int waves, hipStream_t s) {
  return waves == 4   ? launch_grads_most<T, D, MASK, 4>(p, sides, s)
         : waves == 2 ? launch_grads_most<T, D, MASK, 2>(p, sides, s)
                      : launch_grads_most<T, D, MASK, 1>(p, sides, s);
}

// Passes 3 and 4 side by side are faster than one after the other whatever the size: their workgroups fill CUs for each other where
// one pass has too few, and the light end of a triangle goes under the other pass. Four waves on the same rows while that gives one
// workgroup per CU, two as long as the workgroups of 128 rows leave CUs idle (a triangle: or end unevenly), else one. Double-backward, us,
// two launches (the rule before) -> one launch with four | two | one waves on the same rows:
//   fp32 d = 64   2 x 256 67 -> 45 | - | -; 32 x 256 83 -> 66 | 54 | 70; 64 x 256 124 -> 108 | 92 | 83; causal 16 x 1024 382 -> 195 | 166 | 213,
//                 32 x 1024 435 -> 375 | 318 | 296, 32 x 2048 980 -> 1190 | 1034 | 950; no mask 32 x 2048 1808 -> 2186 | 1937 | 1793
//   fp32 d = 128  (one wave at all sizes, LDS) 2 x 256 234 -> 133; causal 16 x 2048 2104 -> 1440; 32 x 2048 2383 -> 2381
//   bf16 d = 32   2 x 256 20 -> 13 | - | -; causal 16 x 1024 99 -> 59 | 47 | 56, 32 x 1024 114 -> 119 | 90 | 96, 64 x 1024 127 -> 218 | 160 | 121
// A side that is far shorter than the other has few workgroups with a long stream each, which nothing fills up: the two sides go
// apart then (split_grads_waves), each with as many waves on the same rows as it needs by itself. Hessian-vector products (here and in
// fhog_attn_split.hip), us, one launch -> apart, by how many times as many rows one side streams: bf16 d = 32 3.1 times (16 x 512 x 1600) 142 -> 147, 5
// times (8 x 512 x 2560) 178 -> 149, the other way round 194 -> 147, 30 times (4 x 200 x 6000) 413 -> 243; fp32 d = 64 3.1 times 370 -> 393,
// 5 times 740 -> 609, 8 times 897 -> 874. fp32 d = 128, which has one wave at all sizes, 8 times 2260 -> 2373: not there.
template <typename T, int D, int MASK>
hipError_t launch_grads(const Params& p, int sides, hipStream_t s) {
  if (rules::few_rows(p, sizeof(T))) return launch_split_few(p, sides, s);
  const int waves = rules::split_grads_waves(p, sizeof(T));
  if (waves) return launch_grads_side<T, D, MASK>(p, sides, waves, s);
  const int64_t g_q = (int64_t)(p.n_q + 127) / 128 * p.batch, g_k = (int64_t)(p.n_k + 127) / 128 * p.batch;
  hipError_t e = hipSuccess;
  if (sides & 1) e = launch_grads_side<T, D, MASK>(p, 1, rules::waves_of_side(g_q, p.n_k), s);
  if (e == hipSuccess && (sides & 2)) e = launch_grads_side<T, D, MASK>(p, 2, rules::waves_of_side(g_k, p.n_q), s);
  return e;
}

template <typename T, int D>
hipError_t launch_td(const Params& p, int pass, hipStream_t s) {
#define FHOG_SPLIT_PASS(N) (p.causal ? launch_sweep<T, D, N, MASK_BAND>(p, s) : launch_sweep<T, D, N, MASK_NONE>(p, s))
  switch (pass) {
    case FHOG_PASS_DD: return FHOG_SPLIT_PASS(1);
    case FHOG_PASS_B: return FHOG_SPLIT_PASS(2);
    case FHOG_PASS_DQ_DDO: return p.causal ? launch_grads<T, D, MASK_BAND>(p, 1, s) : launch_grads<T, D, MASK_NONE>(p, 1, s);
    case FHOG_PASS_DK_DV: return p.causal ? launch_grads<T, D, MASK_BAND>(p, 2, s) : launch_grads<T, D, MASK_NONE>(p, 2, s);
    case FHOG_PASS_DD_B: return FHOG_SPLIT_PASS(5);
    case kPassGrads: return p.causal ? launch_grads<T, D, MASK_BAND>(p, 3, s) : launch_grads<T, D, MASK_NONE>(p, 3, s);
    default: return hipErrorInvalidValue;
  }
#undef FHOG_SPLIT_PASS
}

template <typename T>
hipError_t launch_t(const Params& p, int pass, hipStream_t s) {
  switch (p.d) {
    case 32: return launch_td<T, 32>(p, pass, s);
    case 64: return launch_td<T, 64>(p, pass, s);
    case 128: return launch_td<T, 128>(p, pass, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_split_pass(const Params& p, int dtype, int pass, hipStream_t s) {
  if (dtype == FHOG_DTYPE_FP32) return launch_t<float>(p, pass, s);
  return dtype == FHOG_DTYPE_FP16 ? launch_t<_Float16>(p, pass, s) : launch_t<__bf16>(p, pass, s);
}

}  // namespace fhog
