"""The rules by which a launch is laid out (fhog_rules.h), compiled for the host and asked about shapes."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")

_PROGRAM = r"""
#include <chrono>
#include <cstdio>
#include <cstring>
#include "fhog_rules.h"
namespace fhog {
const Tuning& tuning() { static const Tuning t; return t; }
}
using namespace fhog;
int main() {
  char what[32];
  fhog_bwdbwd_args a = {};
  long long batch, n_q, n_k, d, window, ws;
  int mask;
  while (scanf("%31s %lld %lld %lld %lld %d %lld %lld", what, &batch, &n_q, &n_k, &d, &mask, &window, &ws) == 8) {
    a.batch = batch, a.n_q = n_q, a.n_k = n_k, a.d = d, a.causal = mask, a.window = window, a.ws_bytes = ws;
    Params p = {};
    p.batch = (int)batch, p.n_q = (int)n_q, p.n_k = (int)n_k, p.d = (int)d, p.causal = mask != 0, p.tile_major = p.tile_major_k = p.causal, p.n_split = p.n_split_k = 1;
    rules::mask_params(mask, window, n_q, n_k, &p.mask_off, &p.window);
    if (!strcmp(what, "joint")) {
      int x, y;
      double best = 1e9;
      for (int i = 0; i < 10; i++) {
        const auto t0 = std::chrono::steady_clock::now();
        rules::joint_splits(&a, p, FHOG_PASS_DQ_DDO, &x, &y);
        const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
        best = us < best ? us : best;
      }
      printf("%d %d %.3f\n", x, y, best);
    } else if (!strcmp(what, "hinted")) {   // splits with the hinted workspace, and with any amount
      int x, y, u, v;
      a.ws_bytes = INT64_MAX;
      rules::joint_splits(&a, p, FHOG_PASS_DQ_DDO, &u, &v);
      a.ws_bytes = (int64_t)rules::workspace_hint(&a, p, FHOG_IMPL_BF16);
      rules::joint_splits(&a, p, FHOG_PASS_DQ_DDO, &x, &y);
      printf("%d %d %d %d\n", x, y, u, v);
    } else if (!strcmp(what, "split_order")) {
      rules::pass_order(&a, kPassGrads, p);
      printf("%d %d\n", p.tile_major, p.tile_major_k);
    } else if (!strcmp(what, "instead")) {
      printf("%d\n", rules::splits_instead(&a, p, FHOG_IMPL_BF16));
    } else if (!strcmp(what, "split")) {   // split products, ws: bytes of an element; first backward and double-backward
      AttnParams f = {};
      f.batch = p.batch, f.n_q = p.n_q, f.n_k = p.n_k, f.d = p.d, f.causal = p.causal, f.mask_off = p.mask_off, f.window = p.window;
      printf("%d %d\n", rules::split_bwd_waves(f, (int)ws), rules::split_grads_waves(p, (int)ws));
    } else if (!strcmp(what, "company")) {   // workgroups of the first backward on a CU, and whether its sweeps take turns
      AttnParams f = {};
      f.batch = p.batch, f.n_q = p.n_q, f.n_k = p.n_k, f.d = p.d, f.causal = p.causal, f.mask_off = p.mask_off, f.window = p.window;
      printf("%d\n", (int)rules::bwd_company(f));
    } else if (!strcmp(what, "small")) {   // waves on the same rows: forward, first backward, double-backward
      using rules::Small;
      for (Small w : {Small::forward, Small::backward, Small::double_backward}) printf("%d ", rules::small_waves(w, batch, n_q, n_k, d, mask, window));
      printf("\n");
    } else if (!strcmp(what, "few")) {   // passes 3 and 4 with one output to a workgroup, ws: bytes of an element
      printf("%d\n", rules::few_rows(p, (int)ws));
    } else if (!strcmp(what, "in_turn")) {   // both sweeps of split products tile by tile; two workgroups of the forward on a CU
      const int64_t gq = (n_q + 127) / 128 * batch, gk = (n_k + 127) / 128 * batch;
      printf("%d %d\n", rules::split_in_turn(p, gq, gk), rules::two_forwards_on_a_cu(gq, p.causal));
    } else if (!strcmp(what, "order")) {   // of passes 3 and 4 in one launch
      rules::joint_splits(&a, p, FHOG_PASS_DQ_DDO, &p.n_split, &p.n_split_k);
      rules::grads_order(&a, true, true, p);
      printf("%d %d\n", p.tile_major, p.tile_major_k);
    }
  }
}
"""
NONE, CAUSAL, BOTTOM_RIGHT = range(3)
PLENTY = 1 << 40


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rules")
    (folder / "rules.hip").write_text(_PROGRAM)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", f"-I{ROOT}/include", f"-I{ROOT}/flash-hob_amd/csrc",
                        str(folder / "rules.hip"), "-o", str(folder / "rules")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]

    def some(queries):
        r = subprocess.run([str(folder / "rules")], input="".join(" ".join(map(str, q)) + "\n" for q in queries), capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr[-2000:]
        return [[float(x) for x in line.split()] for line in r.stdout.splitlines()]

    def one(*query):
        return some([query])[0]
    one.some = some
    return one


@pytest.mark.parametrize("mask", [NONE, BOTTOM_RIGHT])
def test_host_time_does_not_grow_with_the_tensors(ask, mask):
    """2^24 keys beside few queries, which would split: the rule looks at no more tiles than for 2^13 keys."""
    short, long = (ask("joint", 1, 1024, n_k, 64, mask, 0, PLENTY)[2] for n_k in (1 << 13, 1 << 24))
    assert long < 10 * short + 5, (short, long)


@pytest.mark.parametrize("shape,splits", [((1, 16384, 16384, 64, NONE, 0), (2, 2)), ((2, 4096, 4096, 64, NONE, 0), (4, 4)), ((1, 8192, 8192, 64, NONE, 0), (4, 4)),
                                          ((2, 8192, 8192, 64, CAUSAL, 0), (4, 4)), ((31, 5588, 980, 64, NONE, 0), (1, 2)), ((8, 2048, 2048, 64, NONE, 0), (1, 1)),
                                          ((2, 8192, 8192, 64, CAUSAL, 500), (1, 1)), ((16, 1000, 3001, 128, BOTTOM_RIGHT, 700), (1, 1))])
def test_splits_of_a_shared_launch(ask, shape, splits):
    """At d = 64 two workgroups share a CU: launches of one workgroup per CU, or of few long ones beside many short ones, split further,
    and those that have company anyway do not. Each pair was measured as the fastest, or within 2 % of it, of all that the rule chooses
    from."""
    assert tuple(ask("joint", *shape, PLENTY)[:2]) == splits


@pytest.mark.parametrize("shape,order", [((1, 19472, 19472, 64, CAUSAL, 0), (1, 1)), ((2, 18809, 18809, 64, CAUSAL, 0), (1, 1)), ((32, 16384, 16384, 64, CAUSAL, 0), (0, 0)),
                                         ((1, 30000, 30000, 64, CAUSAL, 5000), (0, 0)), ((1, 19472, 19472, 128, CAUSAL, 0), (0, 0)), ((2, 9000, 17000, 64, BOTTOM_RIGHT, 0), (1, 1)), ((8, 2000, 17000, 64, BOTTOM_RIGHT, 0), (1, 0)),
                                         ((2, 9000, 17000, 64, BOTTOM_RIGHT, 500), (1, 0)), ((2, 9000, 17000, 128, BOTTOM_RIGHT, 0), (1, 0)),
                                         ((4, 16383, 16383, 128, CAUSAL, 0), (1, 1)), ((1, 20000, 20000, 64, NONE, 0), (0, 0))])
def test_order_of_a_shared_launch(ask, shape, order):
    """Slices of 16384 rows or more go one after the other (0) instead of tile by tile together (1), each side by its own length, except at d = 64 where
    the two sides take turns."""
    assert tuple(ask("order", *shape, PLENTY)) == order


@pytest.mark.parametrize("shape,splits", [((4, 5012, 9866, 64), (2, 1)), ((1, 25434, 25726, 128), (1, 1))])
def test_splits_under_a_mask_give_both_sweeps_as_many_workgroups(ask, shape, splits):
    """us: 4 | 1 splits 524 and 1924, these 471 and 1645."""
    assert tuple(ask("joint", *shape, BOTTOM_RIGHT, 0, PLENTY)[:2]) == splits


@pytest.mark.parametrize("d", [64, 128])
def test_hinted_workspace_has_room_for_both_sides(ask, d):
    """Passes 3 and 4 in one launch hold their partial results at the same time: with the hinted workspace they split as with any amount."""
    lengths = (300, 1000, 1024, 2000, 3000, 4096, 9000, 20000)
    queries = [("hinted", b, n_q, n_k, d, mask, window, 0) for b in (1, 2, 3, 5, 8, 16) for n_q in lengths for n_k in lengths
               for mask, window in ((NONE, 0), (CAUSAL, 0), (BOTTOM_RIGHT, 700)) if mask == NONE or (n_q == n_k if mask == CAUSAL else n_q <= n_k)]
    short = [(q, got) for q, got in zip(queries, ask.some(queries)) if got[:2] != got[2:]]
    assert not short, short[:5]
    if d == 128:   # 38.5 steps of a tile with the room that the wider of the two passes needs, 24 so
        assert ask("hinted", 1, 2000, 1024, 128, NONE, 0, 0)[:2] == [2, 4]


@pytest.mark.parametrize("shape,instead", [((8, 2048, 2048, 64, NONE, 0), 1), ((24, 2048, 2048, 64, NONE, 0), 0), ((16, 2048, 2048, 128, NONE, 0), 0), ((16, 2048, 2048, 64, CAUSAL, 0), 1),
                                           ((4, 8192, 8192, 128, CAUSAL, 0), 1), ((48, 1024, 1024, 64, CAUSAL, 0), 0), ((4, 2048, 2048, 64, CAUSAL, 100), 0), ((1, 17845, 17845, 64, CAUSAL, 5353), 1), ((3, 4096, 4096, 128, CAUSAL, 600), 1),
                                           ((6, 2048, 9000, 64, BOTTOM_RIGHT, 0), 1), ((10, 2048, 9000, 64, BOTTOM_RIGHT, 0), 0)])
def test_schedules_without_a_split_form_are_replaced_where_that_is_faster(ask, shape, instead):
    """By the query side's workgroups of 128 rows under the mask; never without room for partial results."""
    assert ask("instead", *shape, PLENTY) == [instead]
    assert ask("instead", *shape, 0) == [0]


@pytest.mark.parametrize("shape,waves", [((1, 28, 28, 128, NONE, 0), (0, 4, 4)), ((85, 17, 64, 64, NONE, 0), (0, 2, 0)), ((3, 100, 64, 128, NONE, 0), (4, 4, 4)), ((3, 100, 32, 128, NONE, 0), (0, 4, 4)),
                                         ((2, 11806, 12908, 128, BOTTOM_RIGHT, 1530), (0, 0, 0)), ((2, 11806, 12908, 128, BOTTOM_RIGHT, 7000), (2, 0, 0)),
                                         ((2, 8150, 8150, 128, CAUSAL, 3261), (4, 0, 0)), ((1, 11600, 11600, 128, CAUSAL, 2900), (4, 0, 0)), ((1, 11600, 11600, 128, CAUSAL, 6000), (4, 2, 0)),
                                         ((3, 368, 7676, 128, BOTTOM_RIGHT, 3000), (4, 2, 0)), ((1, 15961, 15961, 64, CAUSAL, 4788), (4, 2, 0)), ((2, 15961, 15961, 64, CAUSAL, 4788), (4, 0, 0)), ((1, 26598, 26604, 64, BOTTOM_RIGHT, 7981), (4, 0, 0)),
                                         ((2, 79, 4228, 128, BOTTOM_RIGHT, 1370), (4, 4, 0)), ((1, 1163, 53, 128, NONE, 0), (4, 4, 0)), ((1, 60, 53, 128, NONE, 0), (0, 4, 4)), ((1, 60, 53, 64, NONE, 0), (4, 4, 4)), ((2, 1200, 1200, 128, NONE, 0), (4, 4, 4))])
def test_small_workgroups(ask, shape, waves):
    """Both sides of the lines that windows, few keys and lopsided shapes add to the rule."""
    assert tuple(ask("small", *shape, 0)) == waves


@pytest.mark.parametrize("bytes_,shape,waves", [
    (4, (2, 7490, 2123, 64, NONE, 0), (0, 0)), (4, (4, 2048, 2048, 64, NONE, 0), (2, 2)), (4, (1, 199, 16395, 128, NONE, 0), (0, 2)), (4, (2, 13595, 68, 128, NONE, 0), (0, 1)),
    (4, (32, 2048, 2048, 128, CAUSAL, 0), (0, 1)), (4, (2, 256, 256, 64, NONE, 0), (4, 4)), (2, (64, 1024, 1024, 32, CAUSAL, 0), (1, 1)), (2, (44, 2112, 2112, 32, CAUSAL, 0), (0, 1)),
    (2, (44, 2112, 2112, 32, CAUSAL, 700), (1, 1)), (2, (1, 1799, 96, 32, NONE, 0), (0, 4)), (2, (14, 93, 17, 32, NONE, 0), (4, 4)), (2, (40, 4667, 1344, 32, NONE, 0), (0, 1)),
    (2, (40, 2000, 2000, 32, NONE, 0), (1, 1)), (2, (90, 57, 19, 32, NONE, 0), (2, 1)), (2, (59, 391, 126, 32, NONE, 0), (0, 0)), (2, (2, 2417, 9036, 32, NONE, 0), (2, 0)), (2, (8, 512, 2560, 32, NONE, 0), (0, 0)), (2, (8, 512, 2560, 128, NONE, 0), (0, 0))])
def test_sweeps_of_split_products_in_one_launch_or_apart(ask, bytes_, shape, waves):
    """Waves on the same rows in the shared launch of first backward and double-backward, 0: two launches."""
    assert tuple(ask("split", *shape, bytes_)) == waves


@pytest.mark.parametrize("shape,order", [((2, 9000, 17000, 64, BOTTOM_RIGHT, 0), (1, 0)), ((2, 17000, 17000, 64, CAUSAL, 0), (0, 0)), ((2, 9000, 9000, 32, CAUSAL, 0), (1, 1)),
                                         ((2, 17000, 9000, 32, NONE, 0), (0, 0))])
def test_order_of_a_shared_launch_of_split_products(ask, shape, order):
    assert tuple(ask("split_order", *shape, 0)) == order


@pytest.mark.parametrize("shape,few", [((8, 256, 256, 32, NONE, 0), 1), ((12, 256, 256, 32, NONE, 0), 0), ((8, 512, 512, 32, CAUSAL, 0), 0), ((8, 512, 512, 64, NONE, 0), 1), ((8, 1024, 1024, 64, NONE, 0), 0),
                                       ((16, 256, 256, 64, NONE, 0), 0), ((4, 1024, 1024, 64, CAUSAL, 0), 1), ((8, 1024, 1024, 64, CAUSAL, 0), 0), ((4, 955, 955, 128, NONE, 0), 1), ((5, 955, 955, 128, NONE, 0), 0),
                                       ((5, 955, 955, 128, CAUSAL, 0), 1), ((5, 955, 955, 128, CAUSAL, 500), 0), ((16, 256, 256, 128, NONE, 0), 1), ((32, 256, 256, 128, NONE, 0), 0), ((8, 48, 2858, 128, NONE, 0), 1)])
def test_small_launches_of_fp32_tensors(ask, shape, few):
    """One output to a workgroup in passes 3 and 4, on both sides of the lines; never for 16-bit tensors."""
    assert ask("few", *shape, 4) == [few]
    assert ask("few", *shape, 2) == [0]


@pytest.mark.parametrize("shape,picks", [((64, 1024, 1024, 32, CAUSAL, 0), (1, 0)), ((99, 1024, 1024, 32, CAUSAL, 0), (1, 1)), ((100, 1024, 1024, 32, CAUSAL, 0), (0, 1)), ((64, 1024, 1024, 32, NONE, 0), (0, 1)),
                                         ((64, 1000, 1200, 32, BOTTOM_RIGHT, 0), (0, 0)), ((32, 2000, 2000, 32, CAUSAL, 1200), (1, 0)), ((32, 2000, 2000, 32, CAUSAL, 1199), (0, 0)),
                                         ((150, 450, 450, 32, CAUSAL, 0), (1, 1)), ((150, 449, 449, 32, CAUSAL, 0), (0, 1)), ((106, 384, 384, 32, CAUSAL, 0), (1, 0)), ((107, 384, 384, 32, CAUSAL, 0), (0, 0)), ((150, 256, 256, 32, CAUSAL, 0), (0, 0)),
                                         ((32, 1024, 1024, 64, CAUSAL, 0), (0, 0)), ((32, 1024, 1024, 128, NONE, 0), (0, 0)), ((33, 1024, 1024, 128, NONE, 0), (0, 1)), ((65, 1024, 1024, 128, CAUSAL, 0), (0, 1))])
def test_company_in_launches_of_split_products(ask, shape, picks):
    """Whether the two sweeps take turns (d = 32), and whether two workgroups of the forward share a CU (fp32, d = 128)."""
    assert tuple(ask("in_turn", *shape, 0)) == picks


ALONE, TWO, IN_TURN, THREE = range(4)


@pytest.mark.parametrize("shape,pick", [((29, 1024, 1024, 64, CAUSAL, 0), ALONE), ((30, 1024, 1024, 64, CAUSAL, 0), IN_TURN), ((63, 1024, 1024, 64, CAUSAL, 0), IN_TURN), ((64, 1024, 1024, 64, CAUSAL, 0), TWO),
                                        ((40, 600, 600, 64, CAUSAL, 0), ALONE), ((50, 500, 500, 64, CAUSAL, 0), TWO), ((20, 1024, 1024, 64, CAUSAL, 512), ALONE), ((20, 1024, 1024, 64, CAUSAL, 511), TWO),
                                        ((22, 1000, 1300, 64, BOTTOM_RIGHT, 0), ALONE), ((20, 700, 1400, 64, BOTTOM_RIGHT, 0), TWO), ((16, 1000, 1700, 64, BOTTOM_RIGHT, 600), ALONE),
                                        ((17, 1000, 1700, 64, BOTTOM_RIGHT, 600), TWO), ((16, 1000, 1700, 64, BOTTOM_RIGHT, 300), TWO), ((40, 1100, 1800, 64, BOTTOM_RIGHT, 600), IN_TURN), ((64, 1024, 1024, 64, NONE, 0), TWO),
                                        ((32, 1024, 1024, 32, NONE, 0), TWO), ((33, 1024, 1024, 32, NONE, 0), THREE), ((48, 1024, 1024, 32, NONE, 0), THREE), ((49, 1024, 1024, 32, NONE, 0), TWO),
                                        ((65, 1024, 1024, 32, NONE, 0), THREE), ((33, 1024, 1024, 32, CAUSAL, 0), TWO)])
def test_company_of_the_first_backward(ask, shape, pick):
    """fp32 tensors, one launch for both sweeps with one wave to 32 rows."""
    assert ask("company", *shape, 0) == [pick]
