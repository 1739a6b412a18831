// Rules by which a launch is laid out: splits of the streamed side, order of the workgroups, kernels for small launches. Host code and nothing else.
#pragma once
#include <math.h>

#include "fhog_common.h"

namespace fhog {
namespace rules {

// kernel-side mask parameters: key j is visible to query i iff 0 <= i + off - j < win
inline void mask_params(int32_t causal, int64_t window, int64_t n_q, int64_t n_k, int32_t* off, int32_t* win) {
  *off = causal == FHOG_MASK_BOTTOM_RIGHT ? (int32_t)(n_k - n_q) : 0;
  const int64_t reach = n_q + n_k;  // a window this long hides nothing
  *win = (int32_t)((window == 0 || window > reach) ? reach : window);
}


// ---- splitting the streamed side of small launches (16-bit kernels) -------------------------------------------
// Bytes of d | dd | b, rounded up so that what follows stays 16-byte aligned.
inline size_t stats_bytes(const fhog_bwdbwd_args* a) { return ((size_t)3 * a->batch * a->n_q * sizeof(float) + 15) & ~(size_t)15; }
// fp32 partial results one split of a pass writes
inline size_t split_bytes(const fhog_bwdbwd_args* a, int pass) {
  if (pass == FHOG_PASS_DQ_DDO) return (size_t)2 * a->batch * a->n_q * a->d * sizeof(float);
  if (pass == FHOG_PASS_DK_DV) return (size_t)2 * a->batch * a->n_k * a->d * sizeof(float);
  return (size_t)3 * a->batch * a->n_q * sizeof(float);
}
// Splits a pass would like: enough workgroups for two per CU, every split keeping at least 8 streamed tiles.
inline int wanted_split(const fhog_bwdbwd_args* a, int impl, int pass) {
  if (impl != FHOG_IMPL_BF16 || pass == FHOG_PASS_D || pass > FHOG_PASS_DD_B) return 1;   // passes 6-8 never split
  const bool kside = pass == FHOG_PASS_DK_DV;
  const int64_t groups = ((kside ? a->n_k : a->n_q) + 127) / 128 * a->batch;
  const int64_t streamed = ((kside ? a->n_q : a->n_k) + 31) / 32;
  int s = 1;
  if (!tuning().split) return s;
  while (groups * s < 512 && s < 16 && streamed / (2 * s) >= 8) s *= 2;
  return s;
}
// ... and what of that the workspace has room for
inline int granted_split(const fhog_bwdbwd_args* a, int impl, int pass) {
  int s = wanted_split(a, impl, pass);
  const size_t have = a->ws_bytes > 0 ? (size_t)a->ws_bytes : 0;
  while (s > 1 && stats_bytes(a) + (size_t)s * split_bytes(a, pass) > have) s /= 2;
  return s;
}

// Workgroups (128 stationary rows) of a slice, those with a visible pair, and the tiles that they visit. Of more than 64 workgroups some 64 are looked
// at, evenly spaced: the rule for 1024 queries and 2^24 keys took 235 us of host time with all of them, 0.4 us so.
struct Work {
  double live = 0, sum = 0;
  int64_t groups = 0, longest = 0;
};
template <typename P>   // Params or AttnParams
inline Work work_of(const P& p, bool kside) {
  Work w;
  const int64_t n_sta = kside ? p.n_k : p.n_q, n_str = kside ? p.n_q : p.n_k;
  w.groups = (n_sta + 127) / 128;
  const int64_t step = (w.groups + 63) / 64;
  int64_t seen = 0;
  for (int64_t g = step / 2; g < w.groups; g += step) {
    seen++;
    int64_t lo = 0, hi = n_str;   // streamed rows visible to [r0, r0 + 128)
    if (p.causal) {
      const int64_t r0 = 128 * g;
      const int64_t first = kside ? r0 - p.mask_off : r0 + p.mask_off - p.window + 1;
      const int64_t last = kside ? r0 + 127 - p.mask_off + p.window - 1 : r0 + 127 + p.mask_off;
      lo = first > 0 ? first : 0, hi = last + 1 < n_str ? last + 1 : n_str;
    }
    if (lo >= hi) continue;
    const int64_t tiles = (hi - 1) / 32 - lo / 32 + 1;
    w.live++, w.sum += (double)tiles, w.longest = tiles > w.longest ? tiles : w.longest;
  }
  const double scale = (double)w.groups / (double)seen;
  w.live *= scale, w.sum *= scale;
  return w;
}

// Splits that pass 3 or 4 runs with on its own, of `most`. At d = 128 they keep one workgroup on a CU: what matters there is rounds of 256
// workgroups times the tiles of one, under the mask, and what the partial results cost. In steps of one tile (1.9 us): a
// workgroup needs about 4 to start and to store, combining 2 plus its bytes at 5 TB/s (14.5 us for 66 MB, 8 for 33).
// Where the work of the workgroups differs (causal) the longest one and the average load bound the launch.
// bf16 16 x 1000 x 3001, window 700, us, as many splits as give 512 workgroups -> this rule: pass 3 with 4 -> 2 splits 49.2 + 14.5
// (combining) -> 37.0 + 7.4, pass 4 with 2 -> 1 52.2 + 14.5 -> 56.7. The other passes and d = 64 run two workgroups on a CU.
inline int split_up_to(int most, const fhog_bwdbwd_args* a, const Params& p, int pass) {
  if (most == 1 || a->d != 128 || (pass != FHOG_PASS_DQ_DDO && pass != FHOG_PASS_DK_DV)) return most;
  const Work w = work_of(p, pass == FHOG_PASS_DK_DV);
  if (w.live == 0) return 1;
  int best = 1;
  double best_cost = 0;
  for (int s = 1; s <= most; s *= 2) {
    const double rounds = ceil(w.live * (double)(a->batch * s) / 256), mean = w.sum / w.live;
    const double alone = (double)w.longest / s + 4, load = rounds * (mean / s + 4);
    double cost = alone > load ? alone : load;
    if (s > 1) cost += 2 + (double)s * split_bytes(a, pass) / (5e6 * 1.9);
    if (s == 1 || cost < best_cost) best = s, best_cost = cost;
  }
  return best;
}

inline int launch_split_of(const fhog_bwdbwd_args* a, const Params& p, int impl, int pass) {
  return split_up_to(granted_split(a, impl, pass), a, p, pass);
}

// When the last of n_a jobs of length a and then n_b jobs of length b ends on 256 CUs, each taken by the CU that is free first
inline double makespan(int64_t n_a, double a, int64_t n_b, double b) {
  struct { int64_t cus; double load; } g[32] = {{256, 0}};   // CUs with the same load
  int groups = 1;
  double end = 0;
  for (int side = 0; side < 2; side++) {
    const double length = side ? b : a;
    int64_t n = side ? n_b : n_a;
    if (n >= 1024) {   // all but the last three rounds go to every CU alike
      for (int i = 0; i < groups; i++) g[i].load += length * (double)(n / 256 - 3);
      n -= (n / 256 - 3) * 256;
    }
    while (n > 0) {
      int m = 0;
      for (int i = 1; i < groups; i++)
        if (g[i].load < g[m].load) m = i;
      if (groups == 1 && n >= 512) {   // whole rounds
        g[0].load += length * (double)(n / 256), n %= 256;
      } else if (n >= g[m].cus || groups == 32) {
        n -= g[m].cus, g[m].load += length;
      } else {
        g[groups++] = {n, g[m].load + length};
        g[m].cus -= n, n = 0;
      }
    }
  }
  for (int i = 0; i < groups; i++) end = g[i].load > end ? g[i].load : end;
  return end;
}

// The same with two workgroups on a CU: together they do one step of length 1 (a half each), a workgroup without company takes `alone` for it.
// A CU takes its second workgroup when every other one has its first.
inline double makespan_two(int64_t n_a, double a, int64_t n_b, double b, double alone) {
  struct Cus { int64_t cus; double first, second; } g[64] = {{256, 0, 0}};   // CUs and what is left of their workgroups
  const double kNothing = 1e-9;
  int groups = 1;
  double t = 0;
  int64_t n[2] = {n_a, n_b};
  const double length[2] = {a, b};
  for (int side = 0; side < 2; side++)   // whole rounds: one to three are left of each side
    if (n[side] >= 4 * 512) t += 2 * length[side] * (double)(n[side] / 512 - 3), n[side] -= (n[side] / 512 - 3) * 512;
  for (int steps = 0; steps < 256; steps++) {
    for (int place = 0; place < 2; place++)
      for (int i = 0; i < groups && (n[0] > 0 || n[1] > 0); i++) {
        if (place == 0 ? g[i].first > 0 : g[i].first <= 0 || g[i].second > 0) continue;
        const int side = n[0] > 0 ? 0 : 1;
        if (n[side] < g[i].cus) {
          if (groups == 64) { n[side] = 0; continue; }
          g[groups++] = {g[i].cus - n[side], g[i].first, g[i].second};
          g[i].cus = n[side];
        }
        n[side] -= g[i].cus;
        (place == 0 ? g[i].first : g[i].second) = length[side];
      }
    double next = 0;   // until the first of the workgroups ends
    for (int i = 0; i < groups; i++) {
      if (g[i].first <= 0) continue;
      const double d = g[i].second > 0 ? 2 * (g[i].first < g[i].second ? g[i].first : g[i].second) : alone * g[i].first;
      if (next == 0 || d < next) next = d;
    }
    if (next == 0) break;
    t += next;
    for (int i = 0; i < groups; i++) {
      if (g[i].first <= 0) continue;
      const double done = g[i].second > 0 ? next / 2 : next / alone;
      g[i].first = g[i].first - done > kNothing ? g[i].first - done : 0;
      if (g[i].second > 0) g[i].second = g[i].second - done > kNothing ? g[i].second - done : 0;
      if (g[i].first == 0) g[i].first = g[i].second, g[i].second = 0;
    }
    for (int i = 0; i < groups; i++)   // CUs that have the same left
      for (int k = groups - 1; k > i; k--)
        if (fabs(g[i].first - g[k].first) < kNothing && fabs(g[i].second - g[k].second) < kNothing) g[i].cus += g[k].cus, g[k] = g[--groups];
  }
  return t;
}

// Two sweeps in one launch, Q-tiled and K-tiled, with gq and gk workgroups under a mask: taken in turn, tile by tile, the heaviest of
// both come first and the lightest last; one sweep after the other, the second one's heaviest start when half of the launch is over, or
// join the first one's heaviest on their CUs. From about 1000 workgroups on a side that no longer matters, and the other order keeps fewer
// tensors in an L2 at a time. Double-backward, us, one after the other -> in turn, bf16 causal: d = 64 16 x 2048 148 -> 124, 4 x 8192
// 527 -> 433, 32 x 2048 213 -> 202, 64 x 2048 380 -> 387; d = 128 16 x 2048 188 -> 188, 4 x 8192 651 -> 638, 64 x 2048 675 -> 688.
// At d = 64 sides of unequal length take turns too, unless a window makes their work even, and what the longer one has more (its light end) comes last. us, so:
// bottom-right 2 x 20704 x 20814 1593 -> 1340, 1 x 18029 x 18090 638 -> 547, 2 x 7413 x 8824 345 -> 310; d = 128 16 x 1925 x 3292, window 87 91 -> 100.
inline bool mixed_order(const Params& p, int64_t gq, int64_t gk) {
  const int64_t most = gq > gk ? gq : gk, least = gq + gk - most;
  return p.tile_major && p.tile_major_k && most < 1000 && (gq == gk || (p.d == 64 && most <= 2 * least && 2 * (int64_t)p.window >= p.n_k));
}

constexpr int64_t kMostParts = 2 * 131072 * (int64_t)sizeof(float);   // bytes of partial results per column, at most

// Splits of the two sides where they share a launch, out of those that either would like alone and the workspace has room for. The same
// reckoning in steps of a tile, over the workgroups of both. At d = 128 a CU has one workgroup and a tile takes 1.9 us; at d = 64 two, and
// a tile takes 0.87 us in company and 1.25 times that alone: 256 workgroups there leave every CU half used. us, splits 1 | 1, 2 | 2, 4 | 4, 8 | 8:
// fp16 d = 64 no mask 1 x 8192 369, 232, 203, 211; 1 x 16384 798, 727, 738, 750; 2 x 4096 178, 123, 115, 123; 4 x 4096 208, 203, 211, 229; 8 x 2048 110, 114,
// 123, 142; causal 1 x 16384 683, 611, 499, 439; 2 x 8192 344, 244, 225, 245; 8 x 2048 99, 81, 85, 113. Splits of one side alone at 1 x 16384: 2 | 1 950.
// Over 640 shapes of 1 to 64 slices with 16 to 20000 rows, against the best pair of each: 2.2 % too slow with one workgroup to a CU -> 0.9 %.
// Under a mask the light end of one sweep and the heavy start of the other meet only where both have about as many workgroups: 1000 masked shapes, against
// the best pair of each, without -> with 10 % on pairs beyond 1.5 to 1: d = 64 2.1 % -> 1.7 % too slow, d = 128 1.9 % -> 0.8 %; bottom-right
// d = 64 4 x 5012 x 9866 4 | 1 524, 2 | 1 471, d = 128 1 x 25434 x 25726 4 | 1 1924, 1 | 1 1645.
// q_pass: 3, or 7, which does not split.
inline void joint_splits(const fhog_bwdbwd_args* a, const Params& p, int q_pass, int* s_q, int* s_k) {
  const int most_q = wanted_split(a, FHOG_IMPL_BF16, q_pass), most_k = wanted_split(a, FHOG_IMPL_BF16, FHOG_PASS_DK_DV);
  *s_q = *s_k = 1;
  const int64_t have = a->ws_bytes - (int64_t)stats_bytes(a);
  if ((most_q == 1 && most_k == 1) || have <= 0) return;
  const Work q = work_of(p, false), k = work_of(p, true);
  if (q.live == 0 || k.live == 0) return;
  const bool two = a->d == 64;
  const double fixed = two ? 2 : 4, tile_us = two ? 0.87 : 1.9, alone = 1.25;
  const int64_t bytes_q = (int64_t)split_bytes(a, FHOG_PASS_DQ_DDO), bytes_k = (int64_t)split_bytes(a, FHOG_PASS_DK_DV);
  double best = 0;
  for (int x = 1; x <= most_q; x *= 2)
    for (int y = 1; y <= most_k; y *= 2) {
      const int64_t part = (x > 1 ? x * bytes_q : 0) + (y > 1 ? y * bytes_k : 0);
      if (part > have || part > kMostParts * a->d) continue;
      const double lq = q.sum / q.live / x + fixed, lk = k.sum / k.live / y + fixed;
      const int64_t nq = llround(q.live * (double)(a->batch * x)), nk = llround(k.live * (double)(a->batch * y));
      double cost, longest;   // pass 3 comes first
      if (two) {
        longest = (double)((q.longest + x - 1) / x > (k.longest + y - 1) / y ? (q.longest + x - 1) / x : (k.longest + y - 1) / y) + fixed;
        longest *= nq + nk <= 256 ? alone : 1.5;   // it comes early and has company for half of its way
        cost = makespan_two(nq, lq, nk, lk, alone);
      } else {
        longest = (double)(q.longest / x > k.longest / y ? q.longest / x : k.longest / y) + fixed;
        cost = makespan(nq, lq, nk, lk);
      }
      if (longest > cost) cost = longest;
      if (part > 0) cost += (4 + (double)part / 2.5e6) / tile_us;   // a launch, and the partial results written and read
      const int64_t of_q = q.groups * x, of_k = k.groups * y;
      if (p.causal && 2 * (int64_t)p.window >= a->n_k && (2 * of_q > 3 * of_k || 2 * of_k > 3 * of_q)) cost *= 1.1;
      if ((x == 1 && y == 1) || cost < best) best = cost, *s_q = x, *s_k = y;
    }
}

// Workgroup order within an XCD. With a mask, tile-major (the slices of an XCD advance together, heaviest tiles of all
// of them first) balances the end of a launch; from 16384 stationary rows on a slice alone has tiles enough for that
// and one slice after the other keeps the fetched bytes near the algorithmic ones (measured on N = 16384: 2.2-2.6x
// instead of 4-10x, sweeps b, 3 and 4 0.1-3 % faster, the dd sweep with its three workgroups per CU 4 % slower).
inline bool slice_order(const fhog_bwdbwd_args* a, const Params& p, int64_t rows) { return tuning().order < 0 && p.causal && rows >= 16384; }
// Of a statistics sweep, and of the split products' passes 3 and 4 in whatever launch: each side by its own length
inline void pass_order(const fhog_bwdbwd_args* a, int pass, Params& p) {
  if (pass != FHOG_PASS_DD && slice_order(a, p, a->n_q)) p.tile_major = 0;
  if (slice_order(a, p, a->n_k)) p.tile_major_k = 0;
}
// Of the 16-bit kernels' passes 3 (or 7) and 4, run alone or in a shared launch. d = 64: where the two take turns tile by tile (mixed_order) they do so at any length, unless a
// window makes their work even: one sweep after the other, the second one's heavy tiles come last. Double-backward, us, slice order -> turns (two launches):
// bf16 causal 1 x 17000 612 -> 544 (550), 1 x 35801 2358 -> 2020 (2058), 2 x 18809 1256 -> 1097 (1125); window 5000 1 x 30000 431 -> 440.
inline void grads_order(const fhog_bwdbwd_args* a, bool q_side, bool k_side, Params& p) {
  const int64_t blocks_q = ((a->n_q + 127) / 128 * a->batch * p.n_split + 7) / 8 * 8, blocks_k = ((a->n_k + 127) / 128 * a->batch * p.n_split_k + 7) / 8 * 8;
  if (a->d == 64 && q_side && k_side && 2 * (int64_t)p.window >= a->n_k && mixed_order(p, blocks_q, blocks_k)) return;
  if (slice_order(a, p, a->n_q)) p.tile_major = 0;
  if (slice_order(a, p, a->n_k)) p.tile_major_k = 0;
}

// Workspace with which every pass, run alone, and passes 3 and 4 in a shared launch, whose partial results are there at the same time, have the splits they would like
inline size_t workspace_hint(const fhog_bwdbwd_args* a, const Params& p, int impl) {
  size_t extra = 0;
  for (int pass = FHOG_PASS_DD; pass <= FHOG_PASS_DD_B; pass++) {
    const int s = split_up_to(wanted_split(a, impl, pass), a, p, pass);
    if (s > 1 && (size_t)s * split_bytes(a, pass) > extra) extra = (size_t)s * split_bytes(a, pass);
  }
  if (impl == FHOG_IMPL_BF16) {
    fhog_bwdbwd_args roomy = *a;
    roomy.ws_bytes = INT64_MAX;
    int x, y;
    joint_splits(&roomy, p, FHOG_PASS_DQ_DDO, &x, &y);
    const size_t both = (x > 1 ? x * split_bytes(a, FHOG_PASS_DQ_DDO) : 0) + (y > 1 ? y * split_bytes(a, FHOG_PASS_DK_DV) : 0);
    if (both > extra) extra = both;
  }
  return extra ? stats_bytes(a) + extra : (size_t)3 * a->batch * a->n_q * sizeof(float);
}

// Passes 6, 7 and 8 have no split form. Whether a launch that asks for them is too small and runs the nearest schedule whose passes split instead (three
// sweeps -> fused statistics, ddO early -> four passes), given that the workspace lets pass 3 split: the statistics sweep has the most to gain, whose
// workgroups are the query side's. Time of the schedule asked for over that of the substitute, 1500 shapes, d = 64 | 128, by 128-row groups of queries:
//   no mask    64.. 1.26 | 1.18, 128.. 1.02 | 0.99, 192.. 0.96 | 0.94, 384.. 0.92 | 0.92
//   triangle   64.. 1.73 | 1.55, 128.. 1.36 | 1.25, 192.. 1.12 | 1.08, 256.. 1.04 | 1.02, 384.. 1.01 | 0.99, 512.. 0.94 | 0.93
//   windows of less than half the keys   64.. 0.94 | 1.04, 128.. 0.93 | 0.93, 192.. 0.85 | 0.84; of 512 keys or more, below 96 1.15 | 1.17, 96.. 1.05 | 1.01;
//   of 2048 or more, 140.. 1.2 to 1.3 on single slices of 17000 to 20000 rows
inline bool splits_instead(const fhog_bwdbwd_args* a, const Params& p, int impl) {
  if (granted_split(a, impl, FHOG_PASS_DQ_DDO) == 1) return false;
  const int64_t groups = (a->n_q + 127) / 128 * a->batch;
  if (2 * (int64_t)p.window < a->n_k) return groups < (p.window >= 2048 ? 192 : p.window >= 512 ? 112 : 0);
  return groups < (p.causal && 2 * (int64_t)p.mask_off <= a->n_k ? 384 : 144);
}

// ---- small launches of the 16-bit kernels (fhog_small.hip) ------------------------------------------------------
// Waves that a launch puts on the same 32 stationary rows: 4 or 2, or 0 for the kernels with four waves on 128 rows.
// One workgroup fits a CU: 4 waves as long as that is one round of the 256 CUs (first order, and short streams: 2 waves up to one or two
// rounds where the other kernels would leave CUs idle). `groups` counts 128-row groups of all sides that share a launch, `tiles` the streamed
// tiles of one. A triangle (or a window) is in favour of small workgroups, whose work evens out; the double-backward's other
// kernels split long streams over workgroups (workspace) and win them back there.
// us, other kernels -> 4 waves | 2 waves, square shapes, bf16:
//   forward           d = 64: 64 x 256 9.2 -> 6.5 | 7.4; 8 x 2048 36.7 -> 19.5 | 25.2; causal 32 x 1000 23 -> 16.5 | 17.6
//                     d = 128: 16 x 512 15.7 -> 9.5 | 13.2; 64 x 256 11.0 -> 13.5 | 10.4; 1 x 8192 163 -> 64 | 118
//   first backward    d = 64: 8 x 256 19.0 -> 7.3 | 9.7; 32 x 256 19.4 -> 12.5 | 10.5; 16 x 1024 48 -> 42 | 37; 1 x 8192 303 -> 114 | 152
//                     d = 128: 8 x 256 25 -> 12 | 18; causal 32 x 512 39 -> 41 | 35, no mask 38 -> 51 | 43
//   double-backward   d = 64: 4 x 256 24.1 -> 14.7 | 18.9; 64 x 256 27.2 -> 41 | 30; causal 8 x 1024 46.6 -> 33.8 | 45; 1 x 4096 59 -> 78 | 142
//                     d = 128: 8 x 256 33.3 -> 22.8 | 30.5; 16 x 512 49.7 -> 49.2 | 49.7; causal 3 x 1536 69 -> 62 | 101; 1 x 2048 55 -> 72 | 127
// Windows of less than half the keys leave the work of the workgroups even, so only CUs left idle speak for small ones, and one or two key tiles
// leave three or two of a forward's four waves without one. us, small workgroups -> the other kernels: forward d = 128 1 x 28 5.3 -> 3.9, 4 x 36 5.6 -> 4.8, d = 64 3 x 30
// 4.2 -> 3.4; window 1530 d = 128 2 x 11806 x 12908 65 -> 56; first backward, window 4788 d = 64 2 x 15961 1.25 to 1, window 3261 d = 128 2 x 8150 1.12 to 1.
// The double-backward of d = 128 with few rows on one side and more than 32 tiles for them to stream: 2 x 79 x 4228, window 1370 58 -> 48.
enum class Small { forward, backward, double_backward };
inline int small_waves(Small what, int64_t batch, int64_t n_q, int64_t n_k, int64_t d, int32_t causal, int64_t window) {
  if (tuning().small >= 0) return tuning().small;
  const int64_t g_q = (n_q + 127) / 128 * batch, g_k = (n_k + 127) / 128 * batch;
  // from 256 groups of a side on the kernels with 128 rows fill the GPU
  if (g_q >= 256 || (what != Small::forward && g_k >= 256)) return 0;
  const int64_t off = causal == FHOG_MASK_BOTTOM_RIGHT ? n_k - n_q : 0;
  const bool windowed = causal != FHOG_MASK_NONE && window > 0 && window < n_k, even_window = windowed && 2 * window < n_k;
  const bool uneven = causal != FHOG_MASK_NONE && (windowed || 2 * off <= n_k);
  const int64_t streamed = what == Small::forward || n_k > n_q ? n_k : n_q;
  const int64_t tiles = ((windowed && window + 63 < streamed ? window + 63 : streamed) + 31) / 32;
  if (what == Small::forward) {
    if (n_k <= 32 || (n_k <= 64 && n_q <= (d == 64 ? 40 : 64))) return 0;
    if (g_q <= 64) return 4;
    if (g_q <= 128) return d == 64 || (uneven && tiles >= 32) ? 4 : 2;
    if (tiles < 32) return 0;
    return d == 64 ? (uneven ? 4 : 2) : (uneven && !even_window ? 2 : 0);
  }
  const int64_t groups = g_q + g_k, least = g_q < g_k ? g_q : g_k;
  if (what == Small::backward) {
    if (groups <= 64) return 4;
    if (groups <= 128) return tiles <= 8 ? 2 : 4;
    if (groups <= 256) return d == 64 || (uneven && !(even_window && tiles >= 32 && groups > 160 && least > 64)) ? 2 : 0;
    return d == 64 && uneven && tiles >= 32 && !(even_window && groups > 350) ? 2 : 0;
  }
  if (d == 128 && tiles > 32 && 4 * least < groups - least) return 0;
  if (groups <= 64) return tiles <= (d == 64 ? 64 : 48) ? 4 : 0;
  if (groups <= 128) return tiles <= 8 ? 2 : tiles <= (uneven ? (d == 64 ? 64 : groups <= 96 ? 48 : 32) : d == 64 ? 32 : 16) ? 4 : 0;
  return groups <= 256 && d == 64 && uneven && tiles <= 32 ? 2 : 0;
}
inline int small_waves(Small what, const fhog_attn_args* a) { return small_waves(what, a->batch, a->n_q, a->n_k, a->d, a->causal, a->window); }


// ---- split products: the query-tiled and the key-tiled sweep of a backward pass (fhog_split.hip, fhog_attn_split.hip) ----------------------
// In one launch the two fill CUs for each other; each in a launch of its own (0 below) a side that is far shorter, whose few workgroups have a long
// stream each, gets as many waves on the same rows as it needs by itself. waves_of_side: those, by its 128-row workgroups.
inline int waves_of_side(int64_t groups, int64_t streamed) { return groups < 64 && streamed > 64 ? 4 : groups < 128 && streamed > 32 ? 2 : 1; }
// Whether one side streams four times as many rows as the other
inline bool lopsided(int64_t n_q, int64_t n_k, int64_t window) {
  const int64_t q = n_k < window ? n_k : window, k = n_q < window ? n_q : window;   // rows that a query and a key see, at most
  return q >= 4 * k || k >= 4 * q;
}

// The number of workgroups says what a shared launch gives where the two sides are alike. Where they are not, the two ways are reckoned up, and two
// launches taken where they are clearly shorter. us, one launch by the number of workgroups -> apart: first backward fp32 d = 64 2 x 7490 x 2123 731 -> 383,
// d = 128 1 x 199 x 16395 1776 -> 1235, 2 x 13595 x 68 2141 -> 1621, bf16 d = 32 1 x 7412 x 86 118 -> 88, causal 43 x 3112 291 -> 234; double-backward
// bf16 d = 32 2 x 2417 x 9036 419 -> 303. Of 5400 shapes of 1 to 64 slices with 16 to 20000 rows 186 were more than 3 % slower than with two launches
// and waves_of_side throughout (up to 1.5 times), 63 are (up to 1.15 times).
// What the two ways cost, in steps of one wave's tile of the query side with one wave on 32 rows
struct SplitCost {
  double two, four;           // a step with two and four waves on the same rows
  double key;                 // a step of the key side
  double own, own_waves;      // in a shared launch, where that side takes d = rowsum(O dO) itself: with one and with more waves on the same rows
  double alone;               // a workgroup's step without company, of those that share a CU
  double fixed, launch;       // to start and to store; another launch
  double heaviest;            // how long the longest workgroup has company
  double margin;              // two launches have to be shorter than this part of the shared one
};
constexpr SplitCost kFirstBackward = {1.05, 1.3, 1.25, 1.25, 1.6, 1.3, 0.9, 2.5, 1.65, 0.75}, kDoubleBackward = {1.35, 1.85, 1, 1, 1, 1.07, 2, 3, 1.6, 0.9};

// One launch: the query side (wq waves on the same rows; 0: not in it), then the key side
inline double split_launch(const Work& q, const Work& k, int64_t batch, int wq, int wk, bool two_on_a_cu, const SplitCost& c) {
  const int waves = wq > wk ? wq : wk;
  const bool two = two_on_a_cu && waves == 1;
  const auto length = [&](double tiles, int w, bool key) {
    return tiles / w * (w == 4 ? c.four : w == 2 ? c.two : 1) * (key ? c.key : 1) * (key && wq ? (w == 1 ? c.own : c.own_waves) : 1) + c.fixed;
  };
  const int64_t nq = q.groups * batch * wq, nk = k.groups * batch * wk;
  const double lq = wq ? length(q.sum / (double)q.groups, wq, false) : 0, lk = wk ? length(k.sum / (double)k.groups, wk, true) : 0;
  const double hq = wq ? length((double)((q.longest + wq - 1) / wq * wq), wq, false) : 0, hk = wk ? length((double)((k.longest + wk - 1) / wk * wk), wk, true) : 0;
  const double heaviest = (hq > hk ? hq : hk) * (!two ? 1 : nq + nk <= 256 ? c.alone : c.heaviest);
  const double all = two ? makespan_two(nq, lq, nk, lk, c.alone) : makespan(nq, lq, nk, lk);
  return all > heaviest ? all : heaviest;
}

template <typename P>
inline bool apart_is_faster(const P& p, int waves, int most_waves, bool two_on_a_cu, const SplitCost& c) {
  const Work q = work_of(p, false), k = work_of(p, true);
  const int64_t g_q = q.groups * p.batch, g_k = k.groups * p.batch;
  int wq = waves_of_side(g_q, p.n_k), wk = waves_of_side(g_k, p.n_q);
  wq = wq < most_waves ? wq : most_waves, wk = wk < most_waves ? wk : most_waves;
  return split_launch(q, k, p.batch, wq, 0, two_on_a_cu, c) + split_launch(q, k, p.batch, 0, wk, two_on_a_cu, c) + c.launch <
         c.margin * split_launch(q, k, p.batch, waves, waves, two_on_a_cu, c);
}

// Whether passes 3 and 4 of fp32 tensors run with one output to a workgroup (fhog_split_few.hip). Those workgroups are four to 32 rows of either side, with a third
// more work in all: ahead as long as they are one round of the 256 CUs, and for two where the tiles that a wave streams are what counts, which are
// fewer. At d = 32 a second round is level; under a triangle half of the tiles are not there. Counted are workgroups as long as
// the longest: those of the side that streams fewer rows are shorter by its tiles. Double-backward, us, the other kernels -> these, no mask | causal:
//   d = 32   2 x 256 22.3 -> 19.9 | 22.5 -> 20.3; 4 x 512 34.7 -> 29.7 | 35.1 -> 30.1; beyond: 8 x 512 35.3 -> 41.6 | 35.4 -> 36.8
//   d = 64   2 x 256 44.5 -> 31.3 | 43.8 -> 31.1; 2 x 1024 138 -> 82 | 136 -> 80; 4 x 1024 138 -> 123 | 137 -> 98; 1 x 4096 506 -> 430 | 497 -> 326; beyond:
//            8 x 1024 170 -> 233 | 134 -> 137; two rounds of short streams: 16 x 256 45.2 -> 46.2, 53 x 50 1.2 to 1
//   d = 128  14 x 256 128 -> 107 | 126 -> 91; 4 x 1024 432 -> 362 | 429 -> 292; 2 x 2048 837 -> 702 | 836 -> 555; 1 x 4096 1647 -> 1380 | 1644 -> 1087; beyond:
//            7 x 1024 435 -> 609 | 433 -> 384; 27 x 256 131 -> 179 | 131 -> 130; 2 x 4096 1658 -> 2481 | 1649 -> 1502
// 274 shapes around the lines, of 1 to 56 slices with 32 to 4096 rows: the 131 that this picks take 0.51 to 1.02 times as long, 12 of the others would take
// less than 0.9, most of them triangles with up to a fifth more workgroups than the line.
// The count is that of both sides also where one is launched alone: passes 3 and 4 have the same bits apart.
inline bool few_rows(const Params& p, int bytes) {
  if (bytes != 4) return false;
  if (tuning().few >= 0) return tuning().few;
  const int64_t n_q = p.n_q, n_k = p.n_k, seen = (int64_t)p.window + 31, waves = p.d == 128 ? 2 : 4, fixed = 3;   // to start and to store, in tiles
  const int64_t q = ((n_k < seen ? n_k : seen) + 32 * waves - 1) / (32 * waves) + fixed, k = ((n_q < seen ? n_q : seen) + 32 * waves - 1) / (32 * waves) + fixed;
  const int64_t groups = 2 * ((n_q + 31) / 32 * q + (n_k + 31) / 32 * k) * p.batch / (q > k ? q : k);
  const int64_t longer = n_q > n_k ? n_q : n_k;
  if (groups > 256 && p.d != 128 && (longer < p.window ? longer : p.window) < 320) return false;
  const bool triangle = p.causal && p.window >= p.n_k && 2 * (int64_t)p.mask_off <= p.n_k;
  const int64_t line = p.d == 32 ? 288 : p.d == 64 ? 512 : 576;
  return groups <= (triangle ? line + line / 4 : line);
}

// Both sweeps of a launch of split products at d = 32, gq and gk workgroups of one wave to 32 rows, in turn as in mixed_order: the second one's heavy tiles
// otherwise start when half of the launch is over. Equal sides of fewer than 800 workgroups under a mask that leaves their work uneven. us, one after
// the other -> in turn: double-backward bf16 causal 32 x 1024 104 -> 80, 64 x 1024 137 -> 128, 8 x 4096 440 -> 324, 2 x 17000 1522 -> 1166, window 1200
// 32 x 2000 190 -> 179, fp32 32 x 2048 516 -> 502; training step bf16 64 x 1024 79 -> 75, 8 x 4096 327 -> 281. Not there: 960 workgroups 120 x 900 174 -> 178,
// 1024 225 -> 224, 3072 1559 -> 1611; bottom-right 32 x 1000 x 1500 127 -> 131; window 550 40 x 1000 73 -> 76, 500 32 x 1000 x 3000 82 -> 84; four waves on the
// same rows fp32 16 x 1024 98 -> 106; fp32 d = 64 48 x 1537 889 -> 919, d = 128 32 x 2048 2206 -> 2247, where a CU has one workgroup. Two tiles of rows leave little
// to even out, three or four only launches that end soon: bf16 150 x 256 31 -> 36, 200 x 300 53 -> 57, fp32 198 x 402 189 -> 199; but 87 x 384 42 -> 37, 150 x 450 76 -> 72.
template <typename P>
bool split_in_turn(const P& p, int64_t gq, int64_t gk) {
  return p.d == 32 && p.causal && gq == gk && gq < (p.n_k >= 450 ? 800 : p.n_k > 256 ? 320 : 0) && 5 * (int64_t)p.window >= 3 * (int64_t)p.n_k;
}

// First backward of fp32 tensors, both sweeps in one launch with one wave to 32 rows. d = 64 under a mask: whether two workgroups share a CU, and then whether
// the sweeps take turns. One after the other the heaviest workgroups of both meet on the same CUs. With fewer than two workgroups for every CU a heavy
// one that is joined by another takes nearly as long as both, while other CUs have one: there each has a CU to itself. Short and even ones
// are better off in company at any number. Counted are workgroups that see a row. Training step, us, a CU to each | two, one sweep after the other | two, in turn:
//   causal        10 x 2048 309 | 321 | 325; 17 x 1024 161 | 170 | 171; 30 x 1024 176 | 204 | 179; 3 x 10000 1453 | 1777 | 1594; but 50 x 500 97.7 | 94.3 | 97.4;
//                 from 480 workgroups on 40 x 700 128 | 138 | 121; 8 x 4096 649 | 747 | 640; 12 x 4096 826 | 773 | 730; 31 x 2048 496 | 453 | 438
//   window        500, 5 x 4096 157 | 135 | 135; after other keys with up to 128 workgroups of queries 600, 16 x 1000 x 1700 127 | 143 | 143; 800, 14 x 1000 x 2200 142 | 172 | -;
//                 with more of them 500, 18 x 900 x 1300 142 | 120 | -; 700, 12 x 1500 x 2500 191 | 172 | -; from 480 on 600, 40 x 1100 x 1800 279 | 256 | 231
//   bottom-right  22 x 1000 x 1300 206 | 212 | 191; 20 x 700 x 1400 193 | 167 | 164; 10 x 3000 x 3500 553 | 599 | 523
// d = 32 without a mask: three workgroups on a CU (168 registers) where that saves a part of a round; two, which are 2 to 4 % ahead in whole rounds, elsewhere.
// Two | three: 60 x 500 x 900 130 | 114, 12 x 3000 519 | 499, 24 x 2048 377 | 372, 80 x 1024 293 | 290; but 32 x 1024 127 | 128, 100 x 512 114 | 119, 30 x 1537 314 | 326.
enum class Company { none, two, in_turn, three };
inline Company bwd_company(const AttnParams& p) {
  if (p.d == 32) {
    const int64_t all = ((int64_t)(p.n_q + 127) / 128 + (p.n_k + 127) / 128) * p.batch;
    return !p.causal && ((all > 512 && all <= 768) || all > 1024) ? Company::three : Company::two;
  }
  if (!p.causal) return Company::two;
  const Work q = work_of(p, false), k = work_of(p, true);
  const double groups = (q.live + k.live) * (double)p.batch;
  if (groups >= 480) return groups < 1024 ? Company::in_turn : Company::two;
  const int64_t longest = q.longest < k.longest ? q.longest : k.longest;   // the longest workgroup of either side, in tiles
  if (p.mask_off > 0 && p.window < p.n_k) return q.live * (double)p.batch <= 128 && longest >= 16 ? Company::none : Company::two;
  return longest >= 19 && 4 * (int64_t)p.mask_off <= p.n_k && 2 * (int64_t)p.window >= p.n_k ? Company::none : Company::two;
}

// Forward of fp32 tensors, d = 128: two workgroups on a CU once there are more than one for each, under a mask more than two (a heavy and a light tile
// that share a CU leave the heavy one alone for most of its time). us, one -> two, at so many workgroups: no mask 422 -> 364 (320), 436
// -> 420 (512), 857 -> 816 (1024), but 234 -> 258 (256); causal 324 -> 290 (640), 466 -> 435 (1024), but 235 -> 260 (512).
inline bool two_forwards_on_a_cu(int64_t groups, bool masked) { return groups > (masked ? 512 : 256); }

// Waves on the same 32 rows for passes 3 and 4 in one launch, or 0 for two launches: four waves while that gives one workgroup per CU, two as long as the
// workgroups of 128 rows leave CUs idle (a triangle: or end unevenly), else one. The figures are those of launch_grads (fhog_split.hip).
inline int split_grads_waves(const Params& p, int bytes) {
  const int64_t g_q = (int64_t)(p.n_q + 127) / 128 * p.batch, g_k = (int64_t)(p.n_k + 127) / 128 * p.batch, groups = g_q + g_k;
  const bool triangle = p.causal && (p.window < p.n_k || 2 * (int64_t)p.mask_off <= p.n_k);
  if (bytes * p.d < 512 && groups > 64 && lopsided(p.n_q, p.n_k, p.window)) return 0;
  const int waves = groups <= 64 || (p.d == 32 && triangle && groups <= 128 && p.n_k >= 1024) ? 4 : groups < (triangle ? (p.d == 32 ? 512 : 257) : 160) ? 2 : 1;
  const bool counted = p.d == 32 || (bytes == 4 && p.d == 64);   // 16-bit tensors of d = 64 and 128 were not; d = 128 has one wave at all sizes
  return counted && apart_is_faster(p, waves, 4, p.d == 32, kDoubleBackward) ? 0 : waves;
}

// ... and for the first backward, whose key side then takes the row sums d itself. The figures are those of launch_bwd (fhog_attn_split.hip).
inline int split_bwd_waves(const AttnParams& p, int bytes) {
  const int64_t g_q = (int64_t)(p.n_q + 127) / 128 * p.batch, g_k = (int64_t)(p.n_k + 127) / 128 * p.batch, groups = g_q + g_k;
  const bool triangle = p.causal && (p.window < p.n_k || 2 * (int64_t)p.mask_off <= p.n_k);
  const bool fp32_128 = bytes * p.d >= 512;   // four waves do not fit the LDS
  if (!fp32_128 && groups > 64 && lopsided(p.n_q, p.n_k, p.window)) return 0;
  int waves = 1;
  if (!fp32_128 && groups <= (triangle && p.n_k >= 1024 ? (p.d == 32 ? 256 : 128) : p.d == 32 ? 128 : 64)) waves = 4;
  else if (groups < (triangle ? (p.d == 32 ? 512 : 257) : p.d == 32 ? 320 : 129)) waves = 2;
  if (waves == 1 && p.d > 32) {
    const int64_t rounds = (groups + 255) / 256, apart = (g_q + 255) / 256 + (g_k + 255) / 256;
    if (triangle ? groups >= (p.n_k >= 1024 ? 1024 : 512) : 12 * apart < 13 * rounds) return 0;
  }
  if (bytes == 4) return apart_is_faster(p, waves, fp32_128 ? 2 : 4, p.d == 32, kFirstBackward) ? 0 : waves;
  // 16-bit tensors of d = 32, where taking d costs the key side a fifth
  if (p.causal) return waves == 1 && groups >= 1450 && 2 * (int64_t)p.window >= p.n_k && 2 * (int64_t)p.mask_off <= p.n_k ? 0 : waves;
  const int64_t n_q = p.n_q, n_k = p.n_k;
  const bool long_key_side = waves == 4   ? n_q >= 2 * n_k && n_q - n_k >= 740
                             : waves == 2 ? 2 * n_q >= 3 * n_k && n_q - n_k >= 250
                                          : (2 * n_q >= 5 * n_k && n_q - n_k >= 250) || (groups >= 1000 && 4 * n_q >= 5 * n_k);
  return long_key_side ? 0 : waves;
}

}  // namespace rules
}  // namespace fhog
