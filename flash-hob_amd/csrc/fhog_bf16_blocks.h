// The arithmetic of one 32 x 32 block in the single-role 16-bit kernels (gfx950), shared by the kernels that put four waves on 128
// stationary rows (fhog_bf16.hip, fhog_attn.hip) and those that put them on 32 (fhog_small.hip). `stage` holds the streamed tiles
// of the block in LDS; masked, lo, hi: key (or query) 8g + 4h + e of the tile counts iff lo <= 8g + e <= hi.
#pragma once
#include "fhog_bf16_util.h"

namespace fhog {
namespace bf16k {

// One 32-key x 32-query block of a Q-tiled sweep of the double-backward.
template <bool F16, int D, int PASS>
__device__ __forceinline__ void q_block(const char* stage, const int (&aoff)[D / 16], const int (&troff)[D / 32][2],
                                        const bf16x8_t (&Qb)[D / 16], const bf16x8_t (&ddQb)[D / 16], const bf16x8_t (&dOb)[D / 16],
                                        bool masked, int lo, int hi, float c_scale_log2, float l_log2, float scale, float dsum, float dd,
                                        float kc, float& red, float& red_dd, float& red_vdds, float& red_pu, float& red_p,
                                        f32x16_t (&acc_dq)[D / 32], f32x16_t (&acc_ddo)[D / 32]) {
  constexpr int NT = (PASS == 1) ? 2 : 4, TILE = TS * 2 * D, KK = D / 16, NC = D / 32;
  constexpr bool P3 = PASS == 3 || PASS == 7, WITH_DDO = PASS == 3;
  // The products are issued as a stream of NT*KK k-steps (K, then V, ddK, ddV); the elementwise work
  // is cut into small pieces placed right behind the MFMAs of the same wave, where it runs in the
  // shadow of the matrix pipe. LDS operands are fetched PF steps ahead.
  //   K  : S += K Q^T, ddS += K ddQ^T
  //   V  : dP += V dO^T            + P = exp2(S c - L)                       (pass 2)
  //   ddK: ddS += ddK Q^T          + P (pass 1) | v = P u, sums of v and of P (fused; u = dP - d as in pass 2)
  //   ddV: E += ddV dO^T           + acc += P (ddS - dd) u   (pass 2: u = dP - d and E' = E - dd d come from
  //                                  accumulators that start at the row constants; with the tail, acc ends as
  //                                  sum P (E' + (ddS - dd) u) = sum P (E + ddS u - dP dd))
  //                                | acc_dd += P ddS, acc_vdds += v ddS   (fused)
  //   tail: acc += P ddS (pass 1) | acc += P E (pass 2, fused)
  // Pass 3 (d = 64) runs the same stream with the elementwise work of the producer/consumer kernel (dS = P u behind
  // ddK; w = ddS scale - dd, ddP = P w, z = P (w u - dd d - b) behind ddV; dS' = P E + z in the tail), packs the four
  // tiles to 16 bits and goes on to the second-level products.
  constexpr int kTensorOfPhase[4] = {0, PASS == 1 ? 1 : 2, 1, 3};
  constexpr int NSTEP = NT * KK, PF = 2, NB = PF + 1, EPK = 16 / KK;
  f32x16_t s = {0}, dds = {0}, dp = {0}, e = {0}, pv, us, tt;
  if (PASS == 2 || PASS == 5) {   // u = dP - d and E' = E - kc straight from the matrix pipe (in pass 3 this measured slower)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      dp[r] = -dsum;
      if (PASS == 2) e[r] = -kc;
    }
  }
  uint32_t pk_ds[8], pk_ds2[8], pk_ddp[8], pk_p[8];   // PASS 3: packed dS, dS', ddP, P (registers 2i, 2i+1)
  bf16x8_t a[NB];
#pragma unroll
  for (int i = 0; i < PF; i++) a[i] = lds_read128(stage + kTensorOfPhase[i / KK] * TILE, aoff[i % KK]);
#pragma unroll
  for (int i = 0; i < NSTEP; i++) {
    const int ph = (PASS == 1 && i >= KK) ? 2 : i / KK, kk = i % KK, c = i % NB;
    if (i + PF < NSTEP)
      a[(i + PF) % NB] = lds_read128(stage + kTensorOfPhase[(i + PF) / KK] * TILE, aoff[(i + PF) % KK]);
    __builtin_amdgcn_sched_barrier(0);
    if (ph == 0) {
      s = mfma<F16>(a[c], Qb[kk], s);
      dds = mfma<F16>(a[c], ddQb[kk], dds);
    } else if (ph == 1) {
      dp = mfma<F16>(a[c], dOb[kk], dp);
#pragma unroll
      for (int r = EPK * kk; r < EPK * (kk + 1); r++) pv[r] = __builtin_amdgcn_exp2f(s[r] * c_scale_log2 - l_log2);
    } else if (ph == 2) {
      dds = mfma<F16>(a[c], Qb[kk], dds);
      if ((P3 || PASS == 5) && kk == 0 && masked) {
        keep_branch();
#pragma unroll
        for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
      }
#pragma unroll
      for (int r = EPK * kk; r < EPK * (kk + 1); r++) {
        if (PASS == 1) {
          pv[r] = __builtin_amdgcn_exp2f(s[r] * c_scale_log2 - l_log2);
        } else if (P3) {
          dp[r] -= dsum;                           // u
          us[r] = pv[r] * dp[r];                   // dS = P u (scale applied to the accumulator at the end)
        } else if (PASS == 5) {
          us[r] = pv[r] * dp[r];                   // v = P u
          red_pu += us[r];
          red_p += pv[r];
        }
      }
    } else {
      e = mfma<F16>(a[c], dOb[kk], e);
      if (PASS == 2 && kk == 0 && masked) {
        keep_branch();
#pragma unroll
        for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
      }
#pragma unroll
      for (int r = EPK * kk; r < EPK * (kk + 1); r++) {
        if (PASS == 2) {
          red = __builtin_fmaf(pv[r] * __builtin_fmaf(dds[r], scale, -dd), dp[r], red);   // P w u
        } else if (P3) {
          const float w = __builtin_fmaf(dds[r], scale, -dd);
          const float ddp = pv[r] * w;
          tt[r] = pv[r] * __builtin_fmaf(w, dp[r], -kc);   // z = P (w u - kc)
          if (r & 1) {
            if (WITH_DDO) pk_ddp[r / 2] = pack2<F16>(dds[r - 1], ddp);   // dds[r - 1] holds ddP of the even register by now
            pk_ds[r / 2] = pack2<F16>(us[r - 1], us[r]);
            if (WITH_DDO) pk_p[r / 2] = pack2<F16>(pv[r - 1], pv[r]);
          } else if (WITH_DDO) {
            dds[r] = ddp;
          }
        } else {
          red_dd = __builtin_fmaf(pv[r], dds[r], red_dd);
          red_vdds = __builtin_fmaf(us[r], dds[r], red_vdds);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (PASS == 1) {
    if (masked) {
      keep_branch();
#pragma unroll
      for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; r++) red = __builtin_fmaf(pv[r], dds[r], red);   // scale applied once at the end
  } else if (!P3) {
#pragma unroll
    for (int r = 0; r < 16; r++) red = __builtin_fmaf(pv[r], e[r], red);
  } else {
#pragma unroll
    for (int r = 0; r < 16; r += 2)
      pk_ds2[r / 2] = pack2<F16>(__builtin_fmaf(pv[r], e[r], tt[r]), __builtin_fmaf(pv[r + 1], e[r + 1], tt[r + 1]));
    // dQ2^T += ddK^T dS^T + K^T dS'^T ; ddO^T += V^T ddP^T + ddV^T P^T  (stage order K, ddK, V, ddV)
    constexpr int NIT = 2 * NC;
    const auto opnd = [](const uint32_t* pk, int t) {
      return __builtin_bit_cast(bf16x8_t, u32x4_t{pk[4 * t], pk[4 * t + 1], pk[4 * t + 2], pk[4 * t + 3]});
    };
    constexpr int NX = WITH_DDO ? 4 : 2;   // staged tensors the second level reads: K, ddK (, V, ddV)
    bf16x8_t ta[2][NX];
#pragma unroll
    for (int x = 0; x < NX; x++) ta[0][x] = lds_read_tr_pre(stage + troff[0][0], stage + troff[0][1], x * TILE);
    if (WITH_DDO) {
#pragma unroll
      for (int it = 0; it < NIT; it++) {
        const int t = it / NC, cb = it % NC, c = it & 1;
        if (it + 1 < NIT) {
          const int t1 = (it + 1) / NC, cb1 = (it + 1) % NC;
#pragma unroll
          for (int x = 0; x < NX; x++)
            ta[c ^ 1][x] = lds_read_tr_pre(stage + troff[cb1][0], stage + troff[cb1][1], x * TILE + t1 * 16 * 2 * D);
        }
        __builtin_amdgcn_sched_barrier(0);
        acc_dq[cb] = mfma<F16>(ta[c][1], opnd(pk_ds, t), acc_dq[cb]);
        acc_ddo[cb] = mfma<F16>(ta[c][NX - 2], opnd(pk_ddp, t), acc_ddo[cb]);
        acc_dq[cb] = mfma<F16>(ta[c][0], opnd(pk_ds2, t), acc_dq[cb]);
        acc_ddo[cb] = mfma<F16>(ta[c][NX - 1], opnd(pk_p, t), acc_ddo[cb]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // dQ2 alone: two column blocks per round, so that the MFMAs on one accumulator are two instructions apart
      constexpr int NP = NC / 2;
      bf16x8_t tb[2][2][2];   // [buffer][column block of the pair][K | ddK]
      const auto read_tb = [&](int buf, int it) {
        const int t1 = it / NP, cp1 = it % NP;
#pragma unroll
        for (int cl = 0; cl < 2; cl++)
#pragma unroll
          for (int x = 0; x < 2; x++)
            tb[buf][cl][x] = lds_read_tr_pre(stage + troff[2 * cp1 + cl][0], stage + troff[2 * cp1 + cl][1], x * TILE + t1 * 16 * 2 * D);
      };
#pragma unroll
      for (int x = 0; x < 2; x++) tb[0][0][x] = ta[0][x];
#pragma unroll
      for (int x = 0; x < 2; x++) tb[0][1][x] = lds_read_tr_pre(stage + troff[1][0], stage + troff[1][1], x * TILE);
#pragma unroll
      for (int it = 0; it < 2 * NP; it++) {
        const int t = it / NP, cp = it % NP, c = it & 1;
        if (it + 1 < 2 * NP) read_tb(c ^ 1, it + 1);
        __builtin_amdgcn_sched_barrier(0);
        acc_dq[2 * cp] = mfma<F16>(tb[c][0][1], opnd(pk_ds, t), acc_dq[2 * cp]);
        acc_dq[2 * cp + 1] = mfma<F16>(tb[c][1][1], opnd(pk_ds, t), acc_dq[2 * cp + 1]);
        acc_dq[2 * cp] = mfma<F16>(tb[c][0][0], opnd(pk_ds2, t), acc_dq[2 * cp]);
        acc_dq[2 * cp + 1] = mfma<F16>(tb[c][1][0], opnd(pk_ds2, t), acc_dq[2 * cp + 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

// One 32-query x 32-key block of the K-tiled sweep of the double-backward: queries qb.., keys kw.. (the lane's: kj).
template <bool F16, int D, typename Geo>
__device__ __forceinline__ void k_block(const Geo& geo, const char* stage, const int (&aoff)[D / 16], const int (&troff)[D / 32][2],
                                        const bf16x8_t (&Kb)[D / 16], const bf16x8_t (&ddKb)[D / 16], const bf16x8_t (&Vb)[D / 16],
                                        const bf16x8_t (&ddVb)[D / 16], int qb, int kw, int kj, int h, float c_scale_log2, float scale,
                                        f32x16_t (&acc_dk)[D / 32], f32x16_t (&acc_dv)[D / 32]) {
  constexpr int TILE = TS * 2 * D, KK = D / 16, NC = D / 32;
  const float* stat = reinterpret_cast<const float*>(stage + 3 * TILE);
  // five first-level products in one stream of KK k-steps; the three staged operands of step kk + 1 are
  // fetched before the MFMAs of step kk: S = Q K^T, ddS = ddQ K^T + Q ddK^T, dP = dO V^T, E = dO ddV^T
  // register 4g + i belongs to query qb + 8g + 4h + i: its statistics come from the staged arrays. The accumulators
  // of dP and E start at -d and -(dd d + b): u = dP - d and E' = E - dd d - b come straight from the matrix pipe.
  f32x16_t s = {0}, dds = {0}, dp, e;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const f32x4_t md4 = *reinterpret_cast<const f32x4_t*>(stat + 1 * TS + 8 * g + 4 * h);
    const f32x4_t mk4 = *reinterpret_cast<const f32x4_t*>(stat + 3 * TS + 8 * g + 4 * h);
#pragma unroll
    for (int i = 0; i < 4; i++) dp[4 * g + i] = md4[i], e[4 * g + i] = mk4[i];
  }
  bf16x8_t a[2][3];
#pragma unroll
  for (int x = 0; x < 3; x++) a[0][x] = lds_read128(stage + x * TILE, aoff[0]);
#pragma unroll
  for (int kk = 0; kk < KK; kk++) {
    const int c = kk & 1;
    if (kk + 1 < KK) {
#pragma unroll
      for (int x = 0; x < 3; x++) a[c ^ 1][x] = lds_read128(stage + x * TILE, aoff[kk + 1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    s = mfma<F16>(a[c][0], Kb[kk], s);
    dds = mfma<F16>(a[c][1], Kb[kk], dds);
    dp = mfma<F16>(a[c][2], Vb[kk], dp);
    dds = mfma<F16>(a[c][0], ddKb[kk], dds);
    e = mfma<F16>(a[c][2], ddVb[kk], e);
    __builtin_amdgcn_sched_barrier(0);
  }
  f32x16_t pv;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(stat + 0 * TS + 8 * g + 4 * h);
#pragma unroll
    for (int i = 0; i < 4; i++) pv[4 * g + i] = __builtin_amdgcn_exp2f(s[4 * g + i] * c_scale_log2 - l4[i]);
  }
  if (geo.partial(qb, kw)) {  // wave-uniform: the block holds hidden (query, key) pairs (mask edge or tensor end)
    int lo, hi;                // query row 8g + 4h + i of the tile counts iff lo <= 8g + i <= hi
    geo.limits(qb, kj, h, lo, hi);
    keep_branch();
#pragma unroll
    for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
  }
  // dS -> s, dS' -> e, ddP -> dds (in place; scale on dS, dS' is applied to the accumulators at the end)
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const f32x4_t dd4 = *reinterpret_cast<const f32x4_t*>(stat + 2 * TS + 8 * g + 4 * h);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = 4 * g + i;
      const float pr = pv[r];
      dds[r] = pr * __builtin_fmaf(dds[r], scale, -dd4[i]);   // ddP = P (ddS - dd)
      s[r] = pr * dp[r];                                         // dS = P u
      e[r] = __builtin_fmaf(pr, e[r], dds[r] * dp[r]);           // dS' = P (E' + (ddS - dd) u)
    }
  }
  const bf16x8_t op_ds[2] = {pack_operand<F16>(s, 0), pack_operand<F16>(s, 1)};
  const bf16x8_t op_ds2[2] = {pack_operand<F16>(e, 0), pack_operand<F16>(e, 1)};
  const bf16x8_t op_ddp[2] = {pack_operand<F16>(dds, 0), pack_operand<F16>(dds, 1)};
  // dK2^T += ddQ^T dS + Q^T dS' ; dV2^T += dO^T ddP   (stage order Q, ddQ, dO)
  constexpr int NIT = 2 * NC;
  bf16x8_t ta[2][3];
#pragma unroll
  for (int x = 0; x < 3; x++) ta[0][x] = lds_read_tr_pre(stage + troff[0][0], stage + troff[0][1], x * TILE);
#pragma unroll
  for (int it = 0; it < NIT; it++) {
    const int t = it / NC, cb = it % NC, c = it & 1;
    if (it + 1 < NIT) {
      const int t1 = (it + 1) / NC, cb1 = (it + 1) % NC;
#pragma unroll
      for (int x = 0; x < 3; x++)
        ta[c ^ 1][x] = lds_read_tr_pre(stage + troff[cb1][0], stage + troff[cb1][1], x * TILE + t1 * 16 * 2 * D);
    }
    __builtin_amdgcn_sched_barrier(0);
    acc_dk[cb] = mfma<F16>(ta[c][1], op_ds[t], acc_dk[cb]);
    acc_dv[cb] = mfma<F16>(ta[c][2], op_ddp[t], acc_dv[cb]);
    acc_dk[cb] = mfma<F16>(ta[c][0], op_ds2[t], acc_dk[cb]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ---- first order --------------------------------------------------------------------------------------------------------
// acc[cb] += tile^T (columns 32cb..32cb+31) x operand, for both k-steps and all column blocks of the tile
template <bool F16, int D, int NOP>
__device__ __forceinline__ void second_level(const char* const (&tile)[NOP], const int (&troff)[D / 32][2],
                                             const bf16x8_t (&op)[NOP][2], f32x16_t (&acc)[NOP][D / 32]) {
  constexpr int NC = D / 32, NIT = 2 * NC;
  bf16x8_t a[2][NOP];
#pragma unroll
  for (int x = 0; x < NOP; x++) a[0][x] = lds_read_tr_pre(tile[x] + troff[0][0], tile[x] + troff[0][1], 0);
#pragma unroll
  for (int it = 0; it < NIT; it++) {
    const int t = it / NC, cb = it % NC, c = it & 1;
    if (it + 1 < NIT) {
      const int t1 = (it + 1) / NC, cb1 = (it + 1) % NC;
#pragma unroll
      for (int x = 0; x < NOP; x++)
        a[c ^ 1][x] = lds_read_tr_pre(tile[x] + troff[cb1][0], tile[x] + troff[cb1][1], t1 * 16 * 2 * D);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < NOP; x++) acc[x][cb] = mfma<F16>(a[c][x], op[x][t], acc[x][cb]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// first-level product of one streamed tile with resident rows: out += tile x res^T (streamed rows = M)
template <bool F16, int D, int NRES>
__device__ __forceinline__ void first_level(const char* tile, const int (&aoff)[D / 16], const bf16x8_t* const (&res)[NRES],
                                            f32x16_t (&out)[NRES]) {
  constexpr int KK = D / 16, PF = 2, NB = PF + 1;
  bf16x8_t a[NB];
#pragma unroll
  for (int i = 0; i < PF; i++) a[i] = lds_read128(tile, aoff[i]);
#pragma unroll
  for (int kk = 0; kk < KK; kk++) {
    if (kk + PF < KK) a[(kk + PF) % NB] = lds_read128(tile, aoff[kk + PF]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < NRES; x++) out[x] = mfma<F16>(a[kk % NB], res[x][kk], out[x]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One 32-key x 32-query block of the forward.
template <bool F16, int D>
__device__ __forceinline__ void fwd_block(const char* stage, const int (&aoff)[D / 16], const int (&troff)[D / 32][2],
                                          const bf16x8_t (&Qb)[D / 16], bool masked, int lo, int hi, float c_scale_log2, float& m,
                                          float& l, f32x16_t (&acc)[1][D / 32]) {
  constexpr int TILE = TS * 2 * D, NC = D / 32;
  f32x16_t s[1] = {f32x16_t{0}};
  const bf16x8_t* const res[1] = {Qb};
  first_level<F16, D, 1>(stage, aoff, res, s);  // S^T: s[r] = (key k0 + 8(r/4) + 4h + r%4, query qi)
  f32x16_t x = s[0];   // raw scores; the scale (positive) goes into the exponent's FMA, maxima commute with it
  if (masked) {
    keep_branch();
#pragma unroll
    for (int r = 0; r < 16; r++) x[r] = in_limits(r, lo, hi) ? x[r] : -INFINITY;
  }
  float tmax = fmaxf(fmaxf(x[0], x[1]), x[2]);
#pragma unroll
  for (int r = 3; r < 15; r += 2) tmax = fmaxf(fmaxf(tmax, x[r]), x[r + 1]);
  tmax = fmaxf(tmax, x[15]) * c_scale_log2;
  tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
  // The running maximum follows the row maximum only in jumps of more than kMaxSlack (in log2 units): P may then
  // reach 2^kMaxSlack instead of 1, which costs no precision in a 16-bit float or in the fp32 sums, and the output
  // accumulators are rescaled only in the rare steps where some row jumps (else on about every second tile).
  constexpr float kMaxSlack = 8.f;
  const float m_new = tmax > m + kMaxSlack ? tmax : m;
  // a row whose window starts in a later tile has seen no key yet: keep exp2(-inf - (-inf)) out of it
  const float m_ref = m_new == -INFINITY ? 0.f : m_new;
  const float alpha = __builtin_amdgcn_exp2f(m - m_ref);
  float rs = 0.f;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    x[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(x[r], c_scale_log2, -m_ref));
    rs += x[r];
  }
  l = __builtin_fmaf(l, alpha, rs);
  if (__builtin_amdgcn_ballot_w64(m_new > m) != 0) {  // rescale only when some row's maximum moved
#pragma unroll
    for (int cb = 0; cb < NC; cb++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[0][cb][r] *= alpha;
  }
  m = m_new;
  const bf16x8_t op[1][2] = {{pack_operand<F16>(x, 0), pack_operand<F16>(x, 1)}};
  const char* const vt[1] = {stage + TILE};
  second_level<F16, D, 1>(vt, troff, op, acc);  // O^T += V^T P^T
}

// One 32-key x 32-query block of the Q-tiled first backward (dQ).
template <bool F16, int D>
__device__ __forceinline__ void bwd_q_block(const char* stage, const int (&aoff)[D / 16], const int (&troff)[D / 32][2],
                                            const bf16x8_t (&Qb)[D / 16], const bf16x8_t (&dOb)[D / 16], bool masked, int lo, int hi,
                                            float c_scale_log2, float l_log2, float dsum, f32x16_t (&acc)[1][D / 32]) {
  constexpr int TILE = TS * 2 * D;
  f32x16_t s[1] = {f32x16_t{0}}, dp[1];
#pragma unroll
  for (int r = 0; r < 16; r++) dp[0][r] = -dsum;        // the accumulator ends as dP - d
  const bf16x8_t* const rq[1] = {Qb};
  const bf16x8_t* const rdo[1] = {dOb};
  first_level<F16, D, 1>(stage, aoff, rq, s);           // S^T  = K Q^T
  first_level<F16, D, 1>(stage + TILE, aoff, rdo, dp);  // dP^T = V dO^T - d
  f32x16_t ds;
#pragma unroll
  for (int r = 0; r < 16; r++) ds[r] = __builtin_amdgcn_exp2f(s[0][r] * c_scale_log2 - l_log2) * dp[0][r];
  if (masked) {
    keep_branch();
#pragma unroll
    for (int r = 0; r < 16; r++) ds[r] = in_limits(r, lo, hi) ? ds[r] : 0.f;
  }
  const bf16x8_t op[1][2] = {{pack_operand<F16>(ds, 0), pack_operand<F16>(ds, 1)}};
  const char* const kt[1] = {stage};
  second_level<F16, D, 1>(kt, troff, op, acc);  // dQ^T += K^T dS^T
}

// One 32-query x 32-key block of the K-tiled first backward (dK, dV); L log2(e) and d of the queries behind the staged tiles.
template <bool F16, int D, typename Geo>
__device__ __forceinline__ void bwd_k_block(const Geo& geo, const char* stage, const int (&aoff)[D / 16], const int (&troff)[D / 32][2],
                                            const bf16x8_t (&Kb)[D / 16], const bf16x8_t (&Vb)[D / 16], int qb, int kw, int kj, int h,
                                            float c_scale_log2, f32x16_t (&acc)[2][D / 32]) {
  constexpr int TILE = TS * 2 * D;
  const float* stat = reinterpret_cast<const float*>(stage + 2 * TILE);
  f32x16_t s[1] = {f32x16_t{0}}, dp[1] = {f32x16_t{0}};
  const bf16x8_t* const rk[1] = {Kb};
  const bf16x8_t* const rv[1] = {Vb};
  first_level<F16, D, 1>(stage, aoff, rk, s);           // S  = Q K^T : s[r] = (query qb + 8(r/4) + 4h + r%4, key kj)
  first_level<F16, D, 1>(stage + TILE, aoff, rv, dp);   // dP = dO V^T
  f32x16_t pv, ds;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const f32x4_t l4 = *reinterpret_cast<const f32x4_t*>(stat + 8 * g + 4 * h);
    const f32x4_t d4 = *reinterpret_cast<const f32x4_t*>(stat + TS + 8 * g + 4 * h);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int r = 4 * g + e;
      pv[r] = __builtin_amdgcn_exp2f(s[0][r] * c_scale_log2 - l4[e]);
      ds[r] = dp[0][r] - d4[e];
    }
  }
  if (geo.partial(qb, kw)) {  // wave-uniform: the block holds hidden (query, key) pairs
    int lo, hi;                // query row 8g + 4h + e of the tile counts iff lo <= 8g + e <= hi: it exists and sees key kj
    geo.limits(qb, kj, h, lo, hi);
    keep_branch();
#pragma unroll
    for (int r = 0; r < 16; r++) pv[r] = in_limits(r, lo, hi) ? pv[r] : 0.f;
  }
#pragma unroll
  for (int r = 0; r < 16; r++) ds[r] *= pv[r];
  const bf16x8_t op[2][2] = {{pack_operand<F16>(ds, 0), pack_operand<F16>(ds, 1)}, {pack_operand<F16>(pv, 0), pack_operand<F16>(pv, 1)}};
  const char* const tl[2] = {stage, stage + TILE};
  second_level<F16, D, 2>(tl, troff, op, acc);  // dK^T += Q^T dS ; dV^T += dO^T P
}

}  // namespace bf16k
}  // namespace fhog
