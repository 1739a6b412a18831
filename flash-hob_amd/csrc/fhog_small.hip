// 16-bit kernels for launches too small to fill the GPU (d = 64 and 128): the default schedule of the double-backward in two
// launches (row statistics; dQ2, ddO beside dK2, dV2) and the first-order passes in two (forward; dQ beside dK, dV).
//
// A workgroup is 4 wave64, W = 4 or 2 of them on the SAME 32 stationary rows: each takes every W-th streamed tile, staged by itself
// in LDS of its own, so the sweep has no barrier, and the partial results of the W waves are added through LDS in their order.
// Against four waves on 128 rows that is W times the workgroups with a W-th of the tiles each; every tile is read from L2 once per 32
// rows instead of once per 128. The two tilings of a backward pass do not depend on each other and share a launch: dK and dV need
// d = rowsum(O dO) of the queries that they stream and take it from the staged rows themselves.
//
// What bounds them: latency. One round trip for the resident rows and the first tiles, the blocks of a wave one after the other (0.9 to
// 1.8 us each at d = 128, 0.5 to 1.1 at d = 64), an exchange through LDS and the stores. us, 128-row kernels -> here, bf16 causal:
//   2 x 256   d = 128: forward 11.3 -> 7.2, first backward 25.5 -> 11.6, double-backward 52.0 -> 22.7; d = 64: 8.7 -> 5.4, 20.2 -> 7.2, 39.3 -> 14.9
//   1 x 4096  d = 128: forward 93 -> 33, first backward 187 -> 76; d = 64: 74 -> 23, 160 -> 38
// One wave of such a workgroup keeps a SIMD to itself: at d = 128 the sweeps for dQ2, ddO and dK2, dV2 take 510 registers, which their
// two output accumulators and the resident rows do not leave room to halve.
#include "fhog_bf16_blocks.h"

namespace fhog {
using namespace bf16k;
namespace {

constexpr int WAVES = 4;

__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// 64 lanes x 4 bytes from the lanes' addresses to 256 contiguous bytes of LDS; counted like the loads of Dma
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void stage_words(uint32_t lds, const float* src) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds);
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off\n\t" ::"s"(m0), "v"(src) : "memory", "m0");
}
#pragma clang diagnostic pop

// The streamed tiles of one wave: every W-th one of [begin, end), in a ring of NBUF stages of its own.
// issue(t, lds): requests tile t into the stage at LDS address lds, COUNT loads.
template <int W, int NBUF, int STAGE, int COUNT, typename Issue, typename Block>
__device__ __forceinline__ void own_tiles(int begin, int end, char* ring, const Issue& issue, const Block& block) {
  const uint32_t lds = lds_addr(ring);
  int t = begin;
  bool landed = true;   // first_tiles' requests: every caller has waited for them
  for (int slot = 0; t < end; t += W) {
    if (!landed) {
      // what may still travel is the tile behind this one
      if (NBUF == 2 && t + W < end) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COUNT) : "memory");
      else dma_wait();
    }
    block(ring + slot * STAGE, t);
    lds_reads_done();   // the stage is overwritten next
    if (t + NBUF * W < end) issue(t + NBUF * W, lds + slot * STAGE);
    landed = landed && NBUF == 2 && t == begin;   // the second tile was requested beside the first
    if (NBUF == 2) slot ^= 1;
  }
}
template <int W, int NBUF, int STAGE, typename Issue>
__device__ __forceinline__ void first_tiles(int begin, int end, char* ring, const Issue& issue) {
  if (begin < end) issue(begin, lds_addr(ring));
  if (NBUF == 2 && begin + W < end) issue(begin + W, lds_addr(ring) + STAGE);
}

// Adds the accumulators of the W waves of a row group: its wave ws returns registers 16/W ws .. of every one, four at a time, summed in
// the order of the waves.
template <int W, int NV>
__device__ __forceinline__ void add_waves(const f32x16_t (&acc)[NV], char* smem, int group, int ws, int lane, f32x4_t (&out)[NV][4 / W]) {
  constexpr int G = 4 / W;   // groups of four registers that a wave returns
  f32x4_t* const x = reinterpret_cast<f32x4_t*>(smem) + group * (W * W * NV * G * 64) + lane;
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      x[(((g / G * W + ws) * NV + v) * G + g % G) * 64] = f32x4_t{acc[v][4 * g], acc[v][4 * g + 1], acc[v][4 * g + 2], acc[v][4 * g + 3]};
  __syncthreads();
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int g = 0; g < G; g++) {
      out[v][g] = x[((ws * W * NV + v) * G + g) * 64];
#pragma unroll
      for (int w = 1; w < W; w++) out[v][g] += x[(((ws * W + w) * NV + v) * G + g) * 64];
    }
}
constexpr int add_waves_bytes(int nv) { return 16 * nv * 64 * 16; }

// The columns of a row whose registers add_waves returned: 32 cb + 8 (G ws + g) + 4 h .. + 3, from out[cb][g]
template <bool F16, int NC, int G>
__device__ __forceinline__ void store_part(uint16_t* row, const f32x4_t (*out)[G], float scale, int ws, int h) {
#pragma unroll
  for (int cb = 0; cb < NC; cb++)
#pragma unroll
    for (int g = 0; g < G; g++)
      *reinterpret_cast<u32x2_t*>(row + 32 * cb + 8 * (G * ws + g) + 4 * h) =
          pack4<F16>(out[cb][g][0] * scale, out[cb][g][1] * scale, out[cb][g][2] * scale, out[cb][g][3] * scale);
}

template <int D>
__device__ __forceinline__ void lane_offsets(int lane, int (&aoff)[D / 16], int (&troff)[D / 32][2]) {
#pragma unroll
  for (int kk = 0; kk < D / 16; kk++) aoff[kk] = tile_off<D>(lane & 31, 2 * kk + (lane >> 5));
#pragma unroll
  for (int cb = 0; cb < D / 32; cb++) troff[cb][0] = tr_lane_off_acc<D>(cb, 0, lane), troff[cb][1] = tr_lane_off_acc<D>(cb, 1, lane);
}

template <bool F16, int D>
__device__ __forceinline__ float half_row_dot(const bf16x8_t (&a)[D / 16], const bf16x8_t (&b)[D / 16]) {
  float sum = 0.f;
#pragma unroll
  for (int kk = 0; kk < D / 16; kk++)
#pragma unroll
    for (int e = 0; e < 8; e++) sum = __builtin_fmaf(to_f32<F16>(a[kk][e]), to_f32<F16>(b[kk][e]), sum);
  return sum;
}

// Stages of a wave's ring: as many as let four waves stay within the 160 KiB of a CU
template <int D, int NT>
constexpr int n_buffers = 2 * WAVES * NT * TS * 2 * D <= 128 * 1024 ? 2 : 1;

// ---- double-backward: d, dd, b ------------------------------------------------------------------------------------------
template <int D>
constexpr int stats_lds = WAVES * n_buffers<D, 4> * 4 * TS * 2 * D;

template <bool F16, int D, int MASK, int W>
__global__ void __launch_bounds__(256, 2) small_stats(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int KK = D / 16, NC = D / 32, ROWS = TS * WAVES / W, NT = 4, TILE = TS * 2 * D, STAGE = NT * TILE, NBUF = n_buffers<D, NT>;
  int bh, tile;
  if (!decode_block<MASK>((p.n_q + ROWS - 1) / ROWS, p.batch, MASK != MASK_NONE, p.tile_major, bh, tile)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave / W, ws = wave % W;   // row group of the wave, and which of its streamed tiles it takes
  const int n = lane & 31, h = lane >> 5;
  const int q0 = tile * ROWS + TS * group, qi = q0 + n, qr = min(qi, p.n_q - 1);   // queries past the end compute on a copy of the last row
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb, row = (int64_t)bh * p.n_q + qr;
  const __bf16* const src[NT] = {(const __bf16*)p.k + koff, (const __bf16*)p.ddk + koff, (const __bf16*)p.v + koff, (const __bf16*)p.ddv + koff};

  const StreamKeys<MASK> geo(p.mask_off, p.window, p.n_k);
  int j_begin, j_end;
  geo.tile_range(q0, TS, j_begin, j_end);
  Dma<D, 1> dma;
  dma.init(p.stride_kn, 0, lane);
  const auto issue = [&](int j, uint32_t lds) { dma.template issue_all<NT>(lds, TILE, src, (int64_t)j * TS * p.stride_kn, 0, p.n_k - j * TS); };
  char* const ring = smem + wave * NBUF * STAGE;
  first_tiles<W, NBUF, STAGE>(j_begin + ws, j_end, ring, issue);

  bf16x8_t Qb[KK], ddQb[KK], dOb[KK], Ob[KK];
  load_resident<D>(Qb, (const __bf16*)p.q + qoff, p.stride_qn, qr, h);
  load_resident<D>(ddQb, (const __bf16*)p.ddq + qoff, p.stride_qn, qr, h);
  load_resident<D>(dOb, (const __bf16*)p.dO + qoff, p.stride_qn, qr, h);
  load_resident<D>(Ob, (const __bf16*)p.o + qoff, p.stride_qn, qr, h);
  const float l_log2 = p.lse[row] * kLog2e, c_scale_log2 = p.scale * kLog2e;
  float dsum = half_row_dot<F16, D>(Ob, dOb);   // d_i = sum_c O_ic dO_ic (fhog/triton_bwdbwd.py:580)
  dsum += __shfl_xor(dsum, 32);
  wait_vm0();

  int aoff[KK], troff[NC][2];
  lane_offsets<D>(lane, aoff, troff);
  float red[5] = {};   // sum P E, and over keys of P ddS, v ddS, v and P with v = P u
  f32x16_t none[NC];
  own_tiles<W, NBUF, STAGE, NT * Dma<D, 1>::IPT>(j_begin + ws, j_end, ring, issue, [&](const char* stage, int j) {
    const int k0 = j * TS;
    const bool masked = geo.partial(k0, q0);
    int lo = 0, hi = 0;
    if (masked) keep_branch(), geo.limits(k0, qi, h, lo, hi);
    q_block<F16, D, 5>(stage, aoff, troff, Qb, ddQb, dOb, masked, lo, hi, c_scale_log2, l_log2, p.scale, dsum, 0.f, 0.f, red[0], red[1],
                       red[2], red[3], red[4], none, none);
  });
  __syncthreads();   // the stages are no longer read
  float* const x = reinterpret_cast<float*>(smem) + lane;
#pragma unroll
  for (int i = 0; i < 5; i++) x[(wave * 5 + i) * 64] = red[i];
  __syncthreads();
  if (ws != 0) return;
#pragma unroll
  for (int i = 0; i < 5; i++) {
#pragma unroll
    for (int w = 1; w < W; w++) red[i] += x[((wave + w) * 5 + i) * 64];
    red[i] += __shfl_xor(red[i], 32);
  }
  if (h != 0 || qi >= p.n_q) return;
  const float dd = red[1] * p.scale;
  p.ws_d[row] = dsum;
  p.ws_dd[row] = dd;
  p.ws_b[row] = __builtin_fmaf(-dd, __builtin_fmaf(dsum, red[4], red[3]), __builtin_fmaf(p.scale, red[2], red[0]));
}

// ---- double-backward: dQ2, ddO (workgroups [0, q_blocks)) and dK2, dV2 (the others) -----------------------------------------
template <bool F16, int D, int MASK, int W>
__device__ __forceinline__ void grads_q(const Params& p, char* smem) {
  constexpr int KK = D / 16, NC = D / 32, ROWS = TS * WAVES / W, NT = 4, TILE = TS * 2 * D, STAGE = NT * TILE, NBUF = n_buffers<D, NT>;
  int bh, tile;
  if (!decode_block<MASK>((p.n_q + ROWS - 1) / ROWS, p.batch, MASK != MASK_NONE, p.tile_major, bh, tile)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave / W, ws = wave % W;   // row group of the wave, and which of its streamed tiles it takes
  const int n = lane & 31, h = lane >> 5;
  const int q0 = tile * ROWS + TS * group, qi = q0 + n, qr = min(qi, p.n_q - 1);
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb, row = (int64_t)bh * p.n_q + qr;
  const __bf16* const src[NT] = {(const __bf16*)p.k + koff, (const __bf16*)p.ddk + koff, (const __bf16*)p.v + koff, (const __bf16*)p.ddv + koff};

  const StreamKeys<MASK> geo(p.mask_off, p.window, p.n_k);
  int j_begin, j_end;
  geo.tile_range(q0, TS, j_begin, j_end);
  Dma<D, 1> dma;
  dma.init(p.stride_kn, 0, lane);
  const auto issue = [&](int j, uint32_t lds) { dma.template issue_all<NT>(lds, TILE, src, (int64_t)j * TS * p.stride_kn, 0, p.n_k - j * TS); };
  char* const ring = smem + wave * NBUF * STAGE;
  first_tiles<W, NBUF, STAGE>(j_begin + ws, j_end, ring, issue);

  bf16x8_t Qb[KK], ddQb[KK], dOb[KK];
  load_resident<D>(Qb, (const __bf16*)p.q + qoff, p.stride_qn, qr, h);
  load_resident<D>(ddQb, (const __bf16*)p.ddq + qoff, p.stride_qn, qr, h);
  load_resident<D>(dOb, (const __bf16*)p.dO + qoff, p.stride_qn, qr, h);
  const float l_log2 = p.lse[row] * kLog2e, c_scale_log2 = p.scale * kLog2e;
  const float dsum = p.ws_d[row], dd = p.ws_dd[row], kc = __builtin_fmaf(dd, dsum, p.ws_b[row]);
  wait_vm0();

  int aoff[KK], troff[NC][2];
  lane_offsets<D>(lane, aoff, troff);
  f32x16_t acc_dq[NC], acc_ddo[NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc_dq[cb] = f32x16_t{0}, acc_ddo[cb] = f32x16_t{0};
  float none[5] = {};
  own_tiles<W, NBUF, STAGE, NT * Dma<D, 1>::IPT>(j_begin + ws, j_end, ring, issue, [&](const char* stage, int j) {
    const int k0 = j * TS;
    const bool masked = geo.partial(k0, q0);
    int lo = 0, hi = 0;
    if (masked) keep_branch(), geo.limits(k0, qi, h, lo, hi);
    q_block<F16, D, 3>(stage, aoff, troff, Qb, ddQb, dOb, masked, lo, hi, c_scale_log2, l_log2, p.scale, dsum, dd, kc, none[0], none[1],
                       none[2], none[3], none[4], acc_dq, acc_ddo);
  });
  __syncthreads();   // the stages are no longer read
  f32x16_t acc[2 * NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[cb] = acc_dq[cb], acc[NC + cb] = acc_ddo[cb];
  f32x4_t out[2 * NC][4 / W];
  add_waves<W>(acc, smem, group, ws, lane, out);
  if (qi >= p.n_q) return;
  store_part<F16, NC, 4 / W>((uint16_t*)p.dq2 + qoff + (int64_t)qi * p.stride_qn, out, p.scale, ws, h);
  store_part<F16, NC, 4 / W>((uint16_t*)p.ddo + qoff + (int64_t)qi * p.stride_qn, out + NC, 1.f, ws, h);
}

template <int D>
constexpr int grads_k_stage = 3 * TS * 2 * D + 4 * TS * 4;   // Q, ddQ, dO tiles and the statistics of their rows

template <bool F16, int D, int MASK, int W>
__device__ __forceinline__ void grads_k(const Params& p, char* smem, int id) {
  constexpr int KK = D / 16, NC = D / 32, ROWS = TS * WAVES / W, NT = 3, TILE = TS * 2 * D, STAGE = grads_k_stage<D>, NBUF = n_buffers<D, 4>;
  int bh, tile;
  if (!decode_block<MASK>((p.n_k + ROWS - 1) / ROWS, p.batch, false, p.tile_major, bh, tile, false, id)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave / W, ws = wave % W;
  const int n = lane & 31, h = lane >> 5;
  const int k0 = tile * ROWS + TS * group, kj = k0 + n, kr = min(kj, p.n_k - 1);   // keys past the end compute on a copy of the last row
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb, srow = (int64_t)bh * p.n_q;
  const __bf16* const src[NT] = {(const __bf16*)p.q + qoff, (const __bf16*)p.ddq + qoff, (const __bf16*)p.dO + qoff};

  const StreamQueries<MASK> geo(p.mask_off, p.window, p.n_q);
  int t_begin, t_end;
  geo.tile_range(k0, TS, t_begin, t_end);
  Dma<D, 1> dma;
  dma.init(p.stride_qn, 0, lane);
  const auto issue = [&](int t, uint32_t lds) {
    const int64_t q = srow + min(t * TS + n, p.n_q - 1);
    dma.template issue_all<NT>(lds, TILE, src, (int64_t)t * TS * p.stride_qn, 0, p.n_q - t * TS);
    stage_words(lds + NT * TILE, (h ? p.ws_d : p.lse) + q);
    stage_words(lds + NT * TILE + 2 * TS * 4, (h ? p.ws_b : p.ws_dd) + q);
  };
  char* const ring = smem + wave * NBUF * STAGE;
  first_tiles<W, NBUF, STAGE>(t_begin + ws, t_end, ring, issue);

  bf16x8_t Kb[KK], ddKb[KK], Vb[KK], ddVb[KK];
  load_resident<D>(Kb, (const __bf16*)p.k + koff, p.stride_kn, kr, h);
  load_resident<D>(ddKb, (const __bf16*)p.ddk + koff, p.stride_kn, kr, h);
  load_resident<D>(Vb, (const __bf16*)p.v + koff, p.stride_kn, kr, h);
  load_resident<D>(ddVb, (const __bf16*)p.ddv + koff, p.stride_kn, kr, h);
  wait_vm0();
  const float c_scale_log2 = p.scale * kLog2e;
  int aoff[KK], troff[NC][2];
  lane_offsets<D>(lane, aoff, troff);
  f32x16_t acc_dk[NC], acc_dv[NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc_dk[cb] = f32x16_t{0}, acc_dv[cb] = f32x16_t{0};
  own_tiles<W, NBUF, STAGE, NT * Dma<D, 1>::IPT + 2>(t_begin + ws, t_end, ring, issue, [&](char* stage, int t) {
    // L, d, dd, b as they lie in memory -> L log2(e), -d, dd, -(dd d + b)
    float* const stat = reinterpret_cast<float*>(stage + NT * TILE);
    const float l = stat[n], d = stat[TS + n], dd = stat[2 * TS + n], b = stat[3 * TS + n];
    stat[h * TS + n] = h ? -d : l * kLog2e;
    if (h) stat[3 * TS + n] = -__builtin_fmaf(dd, d, b);
    k_block<F16, D>(geo, stage, aoff, troff, Kb, ddKb, Vb, ddVb, t * TS, k0, kj, h, c_scale_log2, p.scale, acc_dk, acc_dv);
  });
  __syncthreads();
  f32x16_t acc[2 * NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[cb] = acc_dk[cb], acc[NC + cb] = acc_dv[cb];
  f32x4_t out[2 * NC][4 / W];
  add_waves<W>(acc, smem, group, ws, lane, out);
  if (kj >= p.n_k) return;
  store_part<F16, NC, 4 / W>((uint16_t*)p.dk2 + koff + (int64_t)kj * p.stride_kn, out, p.scale, ws, h);
  store_part<F16, NC, 4 / W>((uint16_t*)p.dv2 + koff + (int64_t)kj * p.stride_kn, out + NC, 1.f, ws, h);
}

constexpr int max_of(int a, int b) { return a > b ? a : b; }
template <int D>
constexpr int grads_lds = max_of(WAVES * n_buffers<D, 4> * max_of(4 * TS * 2 * D, grads_k_stage<D>), add_waves_bytes(2 * D / 32));

template <bool F16, int D, int MASK, int W>
__global__ void __launch_bounds__(256, D == 64 ? 2 : 1) small_grads(Params p, int q_blocks) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  if ((int)blockIdx.x < q_blocks) grads_q<F16, D, MASK, W>(p, smem);
  else grads_k<F16, D, MASK, W>(p, smem, (int)blockIdx.x - q_blocks);
}

// ---- first order: forward ---------------------------------------------------------------------------------------------------
template <int D>
constexpr int fwd_lds = max_of(WAVES * n_buffers<D, 2> * 2 * TS * 2 * D, add_waves_bytes(D / 32) + WAVES * 2 * 64 * 4);

template <bool F16, int D, int MASK, int W>
__global__ void __launch_bounds__(256, 2) small_fwd(AttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int KK = D / 16, NC = D / 32, ROWS = TS * WAVES / W, NT = 2, TILE = TS * 2 * D, STAGE = NT * TILE, NBUF = n_buffers<D, NT>;
  int bh, tile;
  if (!decode_block<MASK>((p.n_q + ROWS - 1) / ROWS, p.batch, MASK != MASK_NONE, MASK != MASK_NONE, bh, tile)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave / W, ws = wave % W;   // row group of the wave, and which of its streamed tiles it takes
  const int n = lane & 31, h = lane >> 5;
  const int q0 = tile * ROWS + TS * group, qi = q0 + n, qr = min(qi, p.n_q - 1);
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb;
  const __bf16* const src[NT] = {(const __bf16*)p.k + koff, (const __bf16*)p.v + koff};
  const StreamKeys<MASK> geo(p.mask_off, p.window, p.n_k);
  int j_begin, j_end;
  geo.tile_range(q0, TS, j_begin, j_end);
  Dma<D, 1> dma;
  dma.init(p.stride_kn, 0, lane);
  const auto issue = [&](int j, uint32_t lds) { dma.template issue_all<NT>(lds, TILE, src, (int64_t)j * TS * p.stride_kn, 0, p.n_k - j * TS); };
  char* const ring = smem + wave * NBUF * STAGE;
  first_tiles<W, NBUF, STAGE>(j_begin + ws, j_end, ring, issue);
  bf16x8_t Qb[KK];
  load_resident<D>(Qb, (const __bf16*)p.q + qoff, p.stride_qn, qr, h);
  wait_vm0();
  const float c_scale_log2 = p.scale * kLog2e;
  int aoff[KK], troff[NC][2];
  lane_offsets<D>(lane, aoff, troff);
  float m = -INFINITY, l = 0.f;
  f32x16_t acc[1][NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[0][cb] = f32x16_t{0};
  own_tiles<W, NBUF, STAGE, NT * Dma<D, 1>::IPT>(j_begin + ws, j_end, ring, issue, [&](const char* stage, int j) {
    const int k0 = j * TS;
    const bool masked = geo.partial(k0, q0);
    int lo = 0, hi = 0;
    if (masked) keep_branch(), geo.limits(k0, qi, h, lo, hi);
    fwd_block<F16, D>(stage, aoff, troff, Qb, masked, lo, hi, c_scale_log2, m, l, acc);
  });
  __syncthreads();
  // the waves' rows on one maximum; a wave that has seen no key of a row has l = 0 and m = -inf there
  float* const ml = reinterpret_cast<float*>(smem + add_waves_bytes(NC)) + lane;
  ml[wave * 2 * 64] = m, ml[(wave * 2 + 1) * 64] = l;
  __syncthreads();
  float m_all = -INFINITY, l_all = 0.f;
#pragma unroll
  for (int w = group * W; w < group * W + W; w++) m_all = fmaxf(m_all, ml[w * 2 * 64]);
  const float m_ref = m_all == -INFINITY ? 0.f : m_all;
#pragma unroll
  for (int w = group * W; w < group * W + W; w++) l_all = __builtin_fmaf(ml[(w * 2 + 1) * 64], __builtin_amdgcn_exp2f(ml[w * 2 * 64] - m_ref), l_all);
  const float mine = __builtin_amdgcn_exp2f(m - m_ref);
#pragma unroll
  for (int cb = 0; cb < NC; cb++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[0][cb][r] *= mine;
  f32x4_t out[NC][4 / W];
  add_waves<W>(acc[0], smem, group, ws, lane, out);
  l_all += __shfl_xor(l_all, 32);
  if (qi >= p.n_q) return;
  store_part<F16, NC, 4 / W>((uint16_t*)p.o + qoff + (int64_t)qi * p.stride_qn, out, 1.f / l_all, ws, h);
  if (ws == 0 && h == 0) p.lse[(int64_t)bh * p.n_q + qi] = (m_all + __builtin_amdgcn_logf(l_all)) * 0.6931471805599453f;   // v_log_f32 is log2
}

// ---- first order: dQ (workgroups [0, q_blocks)) and dK, dV (the others) ---------------------------------------------------------
template <bool F16, int D, int MASK, int W>
__device__ __forceinline__ void bwd_q(const AttnParams& p, char* smem) {
  constexpr int KK = D / 16, NC = D / 32, ROWS = TS * WAVES / W, NT = 2, TILE = TS * 2 * D, STAGE = NT * TILE, NBUF = n_buffers<D, NT>;
  int bh, tile;
  if (!decode_block<MASK>((p.n_q + ROWS - 1) / ROWS, p.batch, MASK != MASK_NONE, p.tile_major_q != 0, bh, tile)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave / W, ws = wave % W;   // row group of the wave, and which of its streamed tiles it takes
  const int n = lane & 31, h = lane >> 5;
  const int q0 = tile * ROWS + TS * group, qi = q0 + n, qr = min(qi, p.n_q - 1);
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb, row = (int64_t)bh * p.n_q + qr;
  const __bf16* const src[NT] = {(const __bf16*)p.k + koff, (const __bf16*)p.v + koff};
  const StreamKeys<MASK> geo(p.mask_off, p.window, p.n_k);
  int j_begin, j_end;
  geo.tile_range(q0, TS, j_begin, j_end);
  Dma<D, 1> dma;
  dma.init(p.stride_kn, 0, lane);
  const auto issue = [&](int j, uint32_t lds) { dma.template issue_all<NT>(lds, TILE, src, (int64_t)j * TS * p.stride_kn, 0, p.n_k - j * TS); };
  char* const ring = smem + wave * NBUF * STAGE;
  first_tiles<W, NBUF, STAGE>(j_begin + ws, j_end, ring, issue);
  bf16x8_t Qb[KK], dOb[KK], Ob[KK];
  load_resident<D>(Qb, (const __bf16*)p.q + qoff, p.stride_qn, qr, h);
  load_resident<D>(dOb, (const __bf16*)p.dO + qoff, p.stride_qn, qr, h);
  load_resident<D>(Ob, (const __bf16*)p.o + qoff, p.stride_qn, qr, h);
  const float l_log2 = p.lse[row] * kLog2e, c_scale_log2 = p.scale * kLog2e;
  float dsum = half_row_dot<F16, D>(Ob, dOb);
  dsum += __shfl_xor(dsum, 32);
  wait_vm0();
  int aoff[KK], troff[NC][2];
  lane_offsets<D>(lane, aoff, troff);
  f32x16_t acc[1][NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[0][cb] = f32x16_t{0};
  own_tiles<W, NBUF, STAGE, NT * Dma<D, 1>::IPT>(j_begin + ws, j_end, ring, issue, [&](const char* stage, int j) {
    const int k0 = j * TS;
    const bool masked = geo.partial(k0, q0);
    int lo = 0, hi = 0;
    if (masked) keep_branch(), geo.limits(k0, qi, h, lo, hi);
    bwd_q_block<F16, D>(stage, aoff, troff, Qb, dOb, masked, lo, hi, c_scale_log2, l_log2, dsum, acc);
  });
  __syncthreads();
  f32x4_t out[NC][4 / W];
  add_waves<W>(acc[0], smem, group, ws, lane, out);
  if (qi >= p.n_q) return;
  store_part<F16, NC, 4 / W>((uint16_t*)p.dq + qoff + (int64_t)qi * p.stride_qn, out, p.scale, ws, h);
  if (ws == 0 && h == 0) p.ws_d[row] = dsum;
}

template <int D>
constexpr int bwd_k_stage = 3 * TS * 2 * D + 2 * TS * 4;   // Q, dO, O tiles, L log2(e) and d of their rows
template <int D>
constexpr int bwd_k_buffers = 2 * WAVES * bwd_k_stage<D> <= 128 * 1024 ? 2 : 1;

template <bool F16, int D, int MASK, int W>
__device__ __forceinline__ void bwd_k(const AttnParams& p, char* smem, int id) {
  constexpr int KK = D / 16, NC = D / 32, ROWS = TS * WAVES / W, NT = 3, TILE = TS * 2 * D, STAGE = bwd_k_stage<D>, NBUF = bwd_k_buffers<D>;
  int bh, tile;
  if (!decode_block<MASK>((p.n_k + ROWS - 1) / ROWS, p.batch, false, p.tile_major_k != 0, bh, tile, false, id)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave / W, ws = wave % W;
  const int n = lane & 31, h = lane >> 5;
  const int k0 = tile * ROWS + TS * group, kj = k0 + n, kr = min(kj, p.n_k - 1);
  const int64_t qoff = (int64_t)bh * p.stride_qb, koff = (int64_t)bh * p.stride_kb, srow = (int64_t)bh * p.n_q;
  // bwd_k_block reads Q, dO and, behind them, the statistics; O lies at the end of a stage
  const __bf16* const src[2] = {(const __bf16*)p.q + qoff, (const __bf16*)p.dO + qoff};
  const __bf16* const src_o[1] = {(const __bf16*)p.o + qoff};
  constexpr int STAT = 2 * TILE, O = 2 * TILE + 2 * TS * 4;
  const StreamQueries<MASK> geo(p.mask_off, p.window, p.n_q);
  int t_begin, t_end;
  geo.tile_range(k0, TS, t_begin, t_end);
  Dma<D, 1> dma;
  dma.init(p.stride_qn, 0, lane);
  const auto issue = [&](int t, uint32_t lds) {
    const int64_t adv = (int64_t)t * TS * p.stride_qn;
    dma.template issue_all<2>(lds, TILE, src, adv, 0, p.n_q - t * TS);
    dma.template issue_all<1>(lds + O, TILE, src_o, adv, 0, p.n_q - t * TS);
    stage_words(lds + STAT, p.lse + srow + min(t * TS + n, p.n_q - 1));
  };
  char* const ring = smem + wave * NBUF * STAGE;
  first_tiles<W, NBUF, STAGE>(t_begin + ws, t_end, ring, issue);
  bf16x8_t Kb[KK], Vb[KK];
  load_resident<D>(Kb, (const __bf16*)p.k + koff, p.stride_kn, kr, h);
  load_resident<D>(Vb, (const __bf16*)p.v + koff, p.stride_kn, kr, h);
  wait_vm0();
  const float c_scale_log2 = p.scale * kLog2e;
  int aoff[KK], troff[NC][2];
  lane_offsets<D>(lane, aoff, troff);
  f32x16_t acc[2][NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) acc[0][cb] = f32x16_t{0}, acc[1][cb] = f32x16_t{0};
  own_tiles<W, NBUF, STAGE, NT * Dma<D, 1>::IPT + 1>(t_begin + ws, t_end, ring, issue, [&](char* stage, int t) {
    float* const stat = reinterpret_cast<float*>(stage + STAT);
    bf16x8_t Ob[KK], dOb[KK];
#pragma unroll
    for (int kk = 0; kk < KK; kk++) Ob[kk] = lds_read128(stage + O, aoff[kk]), dOb[kk] = lds_read128(stage + TILE, aoff[kk]);
    float d = half_row_dot<F16, D>(Ob, dOb);
    d += __shfl_xor(d, 32);
    const float l = stat[n];
    stat[h * TS + n] = h ? d : l * kLog2e;
    bwd_k_block<F16, D>(geo, stage, aoff, troff, Kb, Vb, t * TS, k0, kj, h, c_scale_log2, acc);
  });
  __syncthreads();
  f32x16_t all[2 * NC];
#pragma unroll
  for (int cb = 0; cb < NC; cb++) all[cb] = acc[0][cb], all[NC + cb] = acc[1][cb];
  f32x4_t out[2 * NC][4 / W];
  add_waves<W>(all, smem, group, ws, lane, out);
  if (kj >= p.n_k) return;
  store_part<F16, NC, 4 / W>((uint16_t*)p.dk + koff + (int64_t)kj * p.stride_kn, out, p.scale, ws, h);
  store_part<F16, NC, 4 / W>((uint16_t*)p.dv + koff + (int64_t)kj * p.stride_kn, out + NC, 1.f, ws, h);
}

template <int D>
constexpr int bwd_lds = max_of(max_of(WAVES * n_buffers<D, 2> * 2 * TS * 2 * D, WAVES * bwd_k_buffers<D> * bwd_k_stage<D>), add_waves_bytes(2 * D / 32));

template <bool F16, int D, int MASK, int W>
__global__ void __launch_bounds__(256, D == 64 ? 2 : 1) small_bwd(AttnParams p, int q_blocks) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  if ((int)blockIdx.x < q_blocks) bwd_q<F16, D, MASK, W>(p, smem);
  else bwd_k<F16, D, MASK, W>(p, smem, (int)blockIdx.x - q_blocks);
}

template <auto Kernel, typename... Args>
hipError_t launch(unsigned grid, int lds, hipStream_t s, Args... args) {
  const hipError_t e = allow_dynamic_lds<Kernel>(lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(Kernel, dim3(grid), dim3(64 * WAVES), lds, s, args...);
  return hipGetLastError();
}

template <int W>
unsigned blocks(int rows, int batch) { return grid_blocks((rows + TS * WAVES / W - 1) / (TS * WAVES / W), batch); }

template <bool F16, int D, int MASK, int W>
hipError_t bwdbwd_d(const Params& p, hipStream_t s) {
  static_assert(stats_lds<D> <= 160 * 1024 && grads_lds<D> <= 160 * 1024, "the stages of four waves have to fit the LDS");
  const unsigned gq = blocks<W>(p.n_q, p.batch), gk = blocks<W>(p.n_k, p.batch);
  const hipError_t e = launch<small_stats<F16, D, MASK, W>>(gq, stats_lds<D>, s, p);
  return e != hipSuccess ? e : launch<small_grads<F16, D, MASK, W>>(gq + gk, grads_lds<D>, s, p, (int)gq);
}

template <bool F16, int D, int MASK, int W>
hipError_t attn_d(const AttnParams& p, bool backward, hipStream_t s) {
  static_assert(fwd_lds<D> <= 160 * 1024 && bwd_lds<D> <= 160 * 1024, "the stages of four waves have to fit the LDS");
  const unsigned gq = blocks<W>(p.n_q, p.batch), gk = blocks<W>(p.n_k, p.batch);
  if (!backward) return launch<small_fwd<F16, D, MASK, W>>(gq, fwd_lds<D>, s, p);
  return launch<small_bwd<F16, D, MASK, W>>(gq + gk, bwd_lds<D>, s, p, (int)gq);
}

}  // namespace

#define FHOG_SMALL_W(FN, F, DD, M, ...) (waves == 4 ? FN<F, DD, M, 4>(__VA_ARGS__) : FN<F, DD, M, 2>(__VA_ARGS__))
#define FHOG_SMALL(FN, F, DD, ...)                                          \
  (mask == MASK_NONE ? FHOG_SMALL_W(FN, F, DD, MASK_NONE, __VA_ARGS__)      \
                     : mask == MASK_CAUSAL ? FHOG_SMALL_W(FN, F, DD, MASK_CAUSAL, __VA_ARGS__) : FHOG_SMALL_W(FN, F, DD, MASK_BAND, __VA_ARGS__))

hipError_t launch_small_bwdbwd(const Params& p, int waves, hipStream_t s) {
  const int mask = mask_mode(p);
  if (p.f16) return p.d == 128 ? FHOG_SMALL(bwdbwd_d, true, 128, p, s) : FHOG_SMALL(bwdbwd_d, true, 64, p, s);
  return p.d == 128 ? FHOG_SMALL(bwdbwd_d, false, 128, p, s) : FHOG_SMALL(bwdbwd_d, false, 64, p, s);
}

hipError_t launch_small_attn(const AttnParams& p, bool backward, int waves, hipStream_t s) {
  const int mask = mask_mode(p);
  if (p.f16) return p.d == 128 ? FHOG_SMALL(attn_d, true, 128, p, backward, s) : FHOG_SMALL(attn_d, true, 64, p, backward, s);
  return p.d == 128 ? FHOG_SMALL(attn_d, false, 128, p, backward, s) : FHOG_SMALL(attn_d, false, 64, p, backward, s);
}
#undef FHOG_SMALL
#undef FHOG_SMALL_W

}  // namespace fhog
