// Device helpers of the split-product kernels (gfx950): contractions of fp32 accuracy on the 16-bit matrix instructions.
//
// An fp32 number is the exact sum of three bf16 numbers (8 significant bits each: 24 in all), a fp16 number of two, and a
// bf16 number is one. A product of two such sums is a sum of bf16 products, each exact in fp32, accumulated in fp32 by
// v_mfma_f32_32x32x16_bf16, which does 16 times the work of v_mfma_f32_32x32x2_f32 per cycle. Six of the nine terms of
// an fp32 product are kept; the three left out are below 2^-24 of it, the rounding of one fp32 addition.
// The S-shaped operands of the second-level products (P, dS, dS', ddP) are fp32 numbers whatever the tensors are, and three
// terms for every tensor type: two carry 16 bits, which shows in sums that cancel.
#pragma once
#include <type_traits>

#include "fhog_bf16_util.h"

namespace fhog {
namespace splitk {
using namespace bf16k;

// How a tensor type meets the matrix instructions.
//   NF   terms of a tensor in the first-level products (tensor x tensor); F16: they are fp16 as they stand
//   N2   bf16 terms of a tensor in the second-level products (tensor x S-shaped operand); NS: terms of that operand
//   LDS1, LDS2   planes of a staged tile when only first-level products read it / when both do; OFF2: first plane of the latter
template <typename T>
struct Terms;
template <>
struct Terms<__bf16> {
  static constexpr int NF = 1, N2 = 1, NS = 3, LDS1 = 1, LDS2 = 1, OFF2 = 0;
  static constexpr bool F16 = false;
};
template <>
struct Terms<_Float16> {
  static constexpr int NF = 1, N2 = 2, NS = 3, LDS1 = 1, LDS2 = 3, OFF2 = 1;
  static constexpr bool F16 = true;
};
template <>
struct Terms<float> {
  static constexpr int NF = 3, N2 = 3, NS = 3, LDS1 = 3, LDS2 = 3, OFF2 = 0;
  static constexpr bool F16 = false;
};

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;

constexpr float kMaxBf16 = 0x1.fep127f;   // the largest finite bf16

// a and b less a packed pair of bf16. With v_perm_b32: after shifts and masks of a pair that it has just made the compiler converts each
// number by itself.
__device__ __forceinline__ void take_out(uint32_t pair, float& a, float& b) {
  a -= __builtin_bit_cast(float, __builtin_amdgcn_perm(pair, pair, 0x01000c0c));
  b -= __builtin_bit_cast(float, __builtin_amdgcn_perm(pair, pair, 0x03020c0c));
}

// (a, b) -> N packed bf16 terms, each the rounded rest of what the ones before left: x = x0 + x1 (+ x2), exactly for N = 3.
// The rest x - x0 is exact in fp32; a two-element dot product against (-1, 0) or (0, -1) takes it without unpacking x0.
// ANY: for numbers of any size, infinities and NaN among them. Every term but the last is held to the largest finite bf16, so that
// no 0 * Inf of a rest reaches the other element of the pair (another column of the output, in second-level operands) and what
// is not finite sits in the last term, which meets the first term of the other operand alone: an infinity keeps its sign, and a
// finite number that bf16 would round to infinity (from 3.396e38 on) stays itself. Two instructions more per pair and term, hence only
// for tensors whose infinities leave outputs finite or decide them (Stager::ANY_FROM). us, without ANY -> so: fp32 2 x 256, d = 64
// 68.1 -> 67.3, Hessian-vector product of fp32 causal 32 x 2048, d = 128 3361 -> 3388; with ANY for all streamed tiles and
// stationary rows 68.4 -> 72.1 and 3303 -> 3572.
// DOT: the rests by the dot product, the fewest instructions; without: two more a pair and term, which unlike it run beside an MFMA under way.
template <int N, bool ANY, bool DOT = true>
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&out)[N]) {
  // The constants are handed over in registers: as the inline operand -1.0, which the compiler uses for the first one, the
  // instruction did not multiply the low element by -1.
  uint32_t c0, c1;
  asm("s_mov_b32 %0, 0xbf80" : "=s"(c0));
  asm("s_mov_b32 %0, 0xbf800000" : "=s"(c1));
  const bf16x2_t first = __builtin_bit_cast(bf16x2_t, c0), second = __builtin_bit_cast(bf16x2_t, c1);
#pragma unroll
  for (int i = 0; i < N; i++) {
    const bool hold = ANY && i + 1 < N;
    const bf16x2_t t = {(__bf16)(hold ? __builtin_amdgcn_fmed3f(a, -kMaxBf16, kMaxBf16) : a), (__bf16)(hold ? __builtin_amdgcn_fmed3f(b, -kMaxBf16, kMaxBf16) : b)};
    out[i] = __builtin_bit_cast(uint32_t, t);
    if (i + 1 < N && DOT) {
      a = __builtin_amdgcn_fdot2_f32_bf16(t, first, a, false);
      b = __builtin_amdgcn_fdot2_f32_bf16(t, second, b, false);
    } else if (i + 1 < N) {
      take_out(out[i], a, b);
    }
  }
}

// Eight numbers split into terms a little at a time, behind MFMAs: at(slot, slots, pair) does what is due behind MFMA `slot` of
// `slots`, pair(i) being numbers 2 i and 2 i + 1. A term and the rests of a pair wait for one another, so the pairs take
// turns. Same terms as split_pair<N, ANY>, whose dot products a lone wave cannot issue while an MFMA of its own is under way (cycles
// per MFMA and what stands behind it: two dot products 55, four 63; four to six other VALU instructions 34 to 40; nothing 33).
template <int N>
struct Splitting {
  u32x4_t terms[N];
  float rest[4][2];

  template <bool ANY = false, typename Pair>
  __device__ __forceinline__ void at(int slot, int slots, Pair pair) {
#pragma unroll
    for (int turn = 0; turn < 2 * N + 2; turn++) {
      if (slot != turn * slots / (2 * N + 2)) continue;
#pragma unroll
      for (int q = 0; q < N; q++) {   // term q of pair turn - 2 q
        const int i = turn - 2 * q;
        if (i < 0 || i >= 4) continue;
        if (q == 0) pair(i, rest[i][0], rest[i][1]);
        const bool hold = ANY && q + 1 < N;
        const bf16x2_t t = {(__bf16)(hold ? __builtin_amdgcn_fmed3f(rest[i][0], -kMaxBf16, kMaxBf16) : rest[i][0]),
                            (__bf16)(hold ? __builtin_amdgcn_fmed3f(rest[i][1], -kMaxBf16, kMaxBf16) : rest[i][1])};
        const uint32_t u = __builtin_bit_cast(uint32_t, t);
        terms[q][i] = u;
        if (q + 1 < N) take_out(u, rest[i][0], rest[i][1]);
      }
    }
  }
  __device__ __forceinline__ bf16x8_t term(int q) const { return __builtin_bit_cast(bf16x8_t, terms[q]); }
};

// Registers 8t .. 8t+7 of an S-shaped fp32 tile as the B operand of second-level k-step t, in N terms.
template <int N, bool DOT = true>
__device__ __forceinline__ void split_operand(const f32x16_t& x, int t, bf16x8_t (&out)[N]) {
  u32x4_t u[N];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    uint32_t w[N];
    split_pair<N, false, DOT>(x[8 * t + 2 * i], x[8 * t + 2 * i + 1], w);
#pragma unroll
    for (int s = 0; s < N; s++) u[s][i] = w[s];
  }
#pragma unroll
  for (int s = 0; s < N; s++) out[s] = __builtin_bit_cast(bf16x8_t, u[s]);
}

// Eight consecutive elements of a row as they lie in memory.
template <typename T>
struct Chunk {
  u32x4_t v[sizeof(T) / 2];
};
template <typename T>
__device__ __forceinline__ Chunk<T> load_chunk(const T* p) {
  Chunk<T> c;
#pragma unroll
  for (int i = 0; i < (int)sizeof(T) / 2; i++) c.v[i] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const char*>(p) + 16 * i);
  return c;
}
template <typename T>
__device__ __forceinline__ float chunk_elem(const Chunk<T>& c, int e) {
  if constexpr (sizeof(T) == 4) {
    const uint32_t bits = c.v[e / 4][e % 4];
    return __builtin_bit_cast(float, bits);
  } else {
    const uint16_t bits = (uint16_t)(c.v[0][e / 2] >> (16 * (e & 1)));
    return (float)__builtin_bit_cast(T, bits);
  }
}
// ... and its terms: FIRST: those of the first-level products (fp16 stays as it is), else the bf16 terms of the second level
template <typename T, bool FIRST, bool ANY, bool DOT = true, int N>
__device__ __forceinline__ void chunk_terms(const Chunk<T>& c, bf16x8_t (&out)[N]) {
  if constexpr (sizeof(T) == 2 && (FIRST || N == 1)) {
    out[0] = __builtin_bit_cast(bf16x8_t, c.v[0]);
  } else {
    u32x4_t u[N];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint32_t w[N];
      split_pair<N, ANY, DOT>(chunk_elem(c, 2 * i), chunk_elem(c, 2 * i + 1), w);
#pragma unroll
      for (int s = 0; s < N; s++) u[s][i] = w[s];
    }
#pragma unroll
    for (int s = 0; s < N; s++) out[s] = __builtin_bit_cast(bf16x8_t, u[s]);
  }
}

// First-level operand of one stationary row: lane (n = lane % 32, h = lane / 32) holds row n, elements 16 kk + 8 h .. + 7.
template <typename T, int D>
__device__ __forceinline__ void load_resident_terms(bf16x8_t (&dst)[D / 16][Terms<T>::NF], const T* base, int64_t ld, int row, int h) {
#pragma unroll
  for (int kk = 0; kk < D / 16; kk++)
    chunk_terms<T, true, true>(load_chunk<T>(base + (int64_t)row * ld + 16 * kk + 8 * h), dst[kk]);
}

// Stationary fp32 operands too many for their terms to stay in registers.
template <typename T, int D>
constexpr bool is_raw = sizeof(T) == 4 && D == 128;

// Stationary operand of a lane: its row's elements 16 kk + 8 h .. + 7 of every k-step, as terms or as they lie in memory. Split
// without ANY: where one of them is not finite, the outputs of its row are not either.
template <typename T, int D>
struct Resident {
  static constexpr int KK = D / 16, NF = Terms<T>::NF;
  typename std::conditional<is_raw<T, D>, Chunk<T>, bf16x8_t[NF]>::type r[KK];
  __device__ __forceinline__ void load(const T* row, int h) {
#pragma unroll
    for (int kk = 0; kk < KK; kk++) {
      const Chunk<T> c = load_chunk<T>(row + 16 * kk + 8 * h);
      if constexpr (is_raw<T, D>) r[kk] = c;
      else chunk_terms<T, true, false>(c, r[kk]);
    }
  }
  __device__ __forceinline__ void terms(int kk, bf16x8_t (&out)[NF]) const {
    if constexpr (is_raw<T, D>) {
      Chunk<T> c = r[kk];
      // splitting is to happen here, tile after tile: hoisted out of the sweep, the terms would be spilled
      asm volatile("" : "+v"(c.v[0]), "+v"(c.v[1]));
      chunk_terms<T, true, false>(c, out);
    } else {
#pragma unroll
      for (int q = 0; q < NF; q++) out[q] = r[kk][q];
    }
  }
};

// The products of two operands in NA and NB terms that are taken, in the order in which they are added up: small ones first.
template <int NA, int NB>
struct TermPairs {
  int n = 0, a[NA * NB] = {}, b[NA * NB] = {};
  constexpr TermPairs() {
    for (int order = NB - 1; order >= 0; order--)
      for (int i = order < NA ? order : NA - 1; i >= 0; i--) a[n] = i, b[n] = order - i, n++;
  }
};
// acc += a b for operands in NF terms each; the small terms first
template <typename T>
__device__ __forceinline__ f32x16_t mma1(f32x16_t acc, const bf16x8_t (&a)[Terms<T>::NF], const bf16x8_t (&b)[Terms<T>::NF]) {
  constexpr int NF = Terms<T>::NF;
#pragma unroll
  for (int order = NF - 1; order >= 0; order--)
#pragma unroll
    for (int i = order; i >= 0; i--) acc = mfma<Terms<T>::F16>(a[i], b[order - i], acc);
  return acc;
}
// acc += a b for a tensor operand in N2 terms and an S-shaped one in NS terms
template <typename T>
__device__ __forceinline__ f32x16_t mma2(f32x16_t acc, const bf16x8_t (&a)[Terms<T>::N2], const bf16x8_t (&b)[Terms<T>::NS]) {
  constexpr int N2 = Terms<T>::N2, NS = Terms<T>::NS;
#pragma unroll
  for (int order = NS - 1; order >= 0; order--)
#pragma unroll
    for (int i = order < N2 ? order : N2 - 1; i >= 0; i--) acc = mfma<false>(a[i], b[order - i], acc);
  return acc;
}

// Staging of NX tensors' 32-row tiles by 256 threads through registers: the global loads of the next tile are issued before
// a step's arithmetic and the split terms written to LDS behind it. Tile planes are 32 rows of D 16-bit elements, swizzled
// in 16-byte chunks (tile_off); plane q of tensor x starts at (x * PLANES + q) * TILE. Rows past the end of a tensor
// are copies of its last row, as in the 16-bit kernels. Tensors from ANY_FROM on are split with ANY: those that leave outputs
// finite (or decide them) where one of their numbers is not.
template <typename T, int D, int NX, bool SECOND, int ANY_FROM, bool DOT = true>
struct Stager {
  static constexpr int PLANES = SECOND ? Terms<T>::LDS2 : Terms<T>::LDS1;
  static constexpr int TILE = TS * 2 * D, BYTES = NX * PLANES * TILE;
  static constexpr int CPR = D / 8;                                // chunks per row
  static constexpr int PER_TENSOR = TS * CPR;                      // 128 (d = 32), 256 or 512 (d = 128)
  static constexpr int XPI = PER_TENSOR < 256 ? 2 : 1;             // tensors per round of 256 threads (a wave's chunks are of one)
  static constexpr int RPT = PER_TENSOR > 256 ? 2 : 1;             // rounds per tensor
  static constexpr int PER = (NX * RPT + XPI - 1) / XPI;
  Chunk<T> c[PER];

  __device__ __forceinline__ static int tensor_of(int i, int tid) { return XPI * i / RPT + (XPI == 2 ? tid >> 7 : 0); }
  __device__ __forceinline__ static int row_of(int i, int tid) { return RPT == 1 ? tid / CPR % TS : tid / CPR + i % RPT * (256 / CPR); }
  // src[x] + row0 rows is the first row of the tile of tensor x
  __device__ __forceinline__ void fetch_chunk(int i, const T* const (&src)[NX], int64_t ld, int row0, int n_rows, int tid) {
    const int x = XPI * i / RPT;
    const T* base = src[x];
    if (XPI == 2 && x + 1 < NX) base = tid >> 7 ? src[x + 1 < NX ? x + 1 : 0] : base;
    if (NX % XPI && tensor_of(i, tid) >= NX) return;
    const uint32_t off = min(row_of(i, tid), n_rows - 1 - row0) * (uint32_t)ld + 8 * (tid % CPR);   // row strides are below 2^24 elements
    c[i] = load_chunk<T>(reinterpret_cast<const T*>(reinterpret_cast<const char*>(base + (int64_t)row0 * ld) + off * (uint32_t)sizeof(T)));
  }
  __device__ __forceinline__ void fetch(const T* const (&src)[NX], int64_t ld, int row0, int n_rows, int tid) {
#pragma unroll
    for (int i = 0; i < PER; i++) fetch_chunk(i, src, ld, row0, n_rows, tid);
  }
  // publish() and, in the room of what it has split, the next fetch(), a little at a time: what is due behind MFMA `slot` of `slots`.
  // fp32 tensors, d >= 64.
  Splitting<Terms<T>::NF> part;
  template <typename Fetch>
  __device__ __forceinline__ void publish_at(char* stage, int tid, int slot, int slots, Fetch fetch_one) {
    static_assert(XPI == 1 && sizeof(T) == 4, "a chunk of a thread is one tensor's");
    const int each = slots / PER, i = slot / each, at = slot % each;
    if (i >= PER) return;
    const auto pair = [&](int p, float& lo, float& hi) { lo = chunk_elem(c[i], 2 * p), hi = chunk_elem(c[i], 2 * p + 1); };
    if (i / RPT >= ANY_FROM) part.template at<true>(at, each - 1, pair);
    else part.template at<false>(at, each - 1, pair);
    if (at == each / 2) fetch_one(i);   // all its pairs are under way
    if (at == each - 1) {
      char* dst = stage + i / RPT * PLANES * TILE + tile_off<D>(row_of(i, tid), tid % CPR);
#pragma unroll
      for (int q = 0; q < Terms<T>::NF; q++) *reinterpret_cast<bf16x8_t*>(dst + q * TILE) = part.term(q);
    }
  }
  __device__ __forceinline__ void publish(char* stage, int tid) const {
#pragma unroll
    for (int i = 0; i < PER; i++) {
      if (NX % XPI && tensor_of(i, tid) >= NX) continue;
      char* dst = stage + tensor_of(i, tid) * PLANES * TILE + tile_off<D>(row_of(i, tid), tid % CPR);
      const bool any = XPI * i / RPT >= ANY_FROM;
      bf16x8_t f[Terms<T>::NF];
      if (any) chunk_terms<T, true, true, DOT>(c[i], f);
      else chunk_terms<T, true, false, DOT>(c[i], f);
#pragma unroll
      for (int q = 0; q < Terms<T>::NF; q++) *reinterpret_cast<bf16x8_t*>(dst + q * TILE) = f[q];
      if constexpr (SECOND && Terms<T>::OFF2 > 0) {
        bf16x8_t s[Terms<T>::N2];
        if (any) chunk_terms<T, false, true>(c[i], s);
        else chunk_terms<T, false, false>(c[i], s);
#pragma unroll
        for (int q = 0; q < Terms<T>::N2; q++) *reinterpret_cast<bf16x8_t*>(dst + (Terms<T>::OFF2 + q) * TILE) = s[q];
      }
    }
  }
};

// First-level A operand of k-step kk from a staged tensor (row = lane % 32): off = tile_off<D>(n, 2 kk + h)
template <typename T, int TILE>
__device__ __forceinline__ void read_terms(const char* tensor, int off, bf16x8_t (&a)[Terms<T>::NF]) {
#pragma unroll
  for (int q = 0; q < Terms<T>::NF; q++) a[q] = lds_read128(tensor + q * TILE, off);
}
// Second-level A operand of k-step t (transposed): o0 / o1 = tr_lane_off_acc<D>(cb, 0 / 1)
template <typename T, int D>
__device__ __forceinline__ void read_terms_tr(const char* tensor, int o0, int o1, int t, bf16x8_t (&a)[Terms<T>::N2]) {
  constexpr int TILE = TS * 2 * D;
#pragma unroll
  for (int q = 0; q < Terms<T>::N2; q++)
    a[q] = lds_read_tr_pre(tensor + o0, tensor + o1, (Terms<T>::OFF2 + q) * TILE + t * 16 * 2 * D);
}

// acc += X^T W for a staged tensor X (32 rows) and an S-shaped tile W whose registers run over those rows
template <typename T, int D, bool DOT = true>
__device__ __forceinline__ void second_level(f32x16_t (&acc)[D / 32], const char* tensor, const int (&troff)[D / 32][2], const f32x16_t& w) {
#pragma unroll
  for (int t = 0; t < 2; t++) {
    bf16x8_t op[Terms<T>::NS];
    split_operand<Terms<T>::NS, DOT>(w, t, op);
#pragma unroll
    for (int cb = 0; cb < D / 32; cb++) {
      bf16x8_t a[Terms<T>::N2];
      read_terms_tr<T, D>(tensor, troff[cb][0], troff[cb][1], t, a);
      acc[cb] = mma2<T>(acc[cb], a, op);
    }
  }
}

// Second-level products one after the other for a lone wave on its SIMD: the LDS operands of a group of products (one k-step, 32 columns)
// are read while the group before is in the matrix pipe, and the next k-step of the S-shaped operand is split behind its
// MFMAs, a pair of numbers at a time. The fences hold the order; left alone, the compiler reads and splits next to the use.
template <typename T, int D>
struct SecondLevel {
  static constexpr int N2 = Terms<T>::N2, NS = Terms<T>::NS, NC = D / 32, TILE = TS * 2 * D;
  static constexpr TermPairs<N2, NS> kPairs{};
  int tr0, tr1;      // tr_lane_off_acc<D>(0, 0 | 1, lane)
  bf16x8_t a[N2];    // operand of the first group to come
  Splitting<NS> op;  // terms of the first k-step to come

  __device__ __forceinline__ void read(const char* tensor, int t, int cb, bf16x8_t (&x)[N2]) const {
    read_terms_tr<T, D>(tensor, tr0 ^ (64 * cb), tr1 ^ (64 * cb), t, x);   // 32 columns are four chunks of 16 bytes
  }
  __device__ __forceinline__ void start(const char* tensor, const f32x16_t& w) {
    read(tensor, 0, 0, a);
    op.at(0, 1, [&](int i, float& lo, float& hi) { lo = w[2 * i], hi = w[2 * i + 1]; });
    __builtin_amdgcn_sched_barrier(0);
  }
  // acc += X^T W for the staged tensor X and the S-shaped tile W whose first operands are at hand; MORE: those of next_w and
  // next_tensor are fetched. work(i): what is to be done behind MFMA i.
  template <bool MORE, typename Work>
  __device__ __forceinline__ void run(f32x16_t (&acc)[NC], const char* tensor, const f32x16_t& w, const char* next_tensor, const f32x16_t& next_w, Work work) {
    constexpr int PER_STEP = NC * kPairs.n;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      Splitting<NS> next_op;
#pragma unroll
      for (int cb = 0; cb < NC; cb++) {
        bf16x8_t next_a[N2];
        const bool step_ends = cb + 1 == NC;
        if (!(step_ends && t == 1)) read(tensor, step_ends ? 1 : t, step_ends ? 0 : cb + 1, next_a);
        else if (MORE) read(next_tensor, 0, 0, next_a);
#pragma unroll
        for (int i = 0; i < kPairs.n; i++) {
          acc[cb] = mfma<false>(a[kPairs.a[i]], op.term(kPairs.b[i]), acc[cb]);
          const int slot = cb * kPairs.n + i;
          if (t == 0 || MORE) next_op.at(slot, PER_STEP, [&](int x, float& lo, float& hi) {
            lo = t == 0 ? w[8 + 2 * x] : next_w[2 * x], hi = t == 0 ? w[9 + 2 * x] : next_w[2 * x + 1];
          });
          work(t * PER_STEP + slot);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (!(step_ends && t == 1) || MORE) {
#pragma unroll
          for (int q = 0; q < N2; q++) a[q] = next_a[q];
        }
      }
      if (t == 0 || MORE) op = next_op;
    }
  }
};

// acc[cb][r] holds column cb*32 + 8*(r/4) + 4*h + r%4 of the lane's stationary row
template <typename T, int D>
__device__ __forceinline__ void store_rows(T* row, const f32x16_t (&acc)[D / 32], float scale, int h) {
#pragma unroll
  for (int cb = 0; cb < D / 32; cb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const float x[4] = {acc[cb][4 * g] * scale, acc[cb][4 * g + 1] * scale, acc[cb][4 * g + 2] * scale, acc[cb][4 * g + 3] * scale};
      T* dst = row + cb * 32 + 8 * g + 4 * h;
      if constexpr (sizeof(T) == 4) *reinterpret_cast<f32x4_t*>(dst) = f32x4_t{x[0], x[1], x[2], x[3]};
      else *reinterpret_cast<u32x2_t*>(dst) = pack4<Terms<T>::F16>(x[0], x[1], x[2], x[3]);
    }
}

}  // namespace splitk
}  // namespace fhog
