"""GPU tier: 16-bit launches too small to fill the GPU, whose four waves work on 32 or 64 stationary rows (fhog_small.hip), against the
kernels with four waves on 128 rows. FHOG_TUNE chooses between them, in one process each."""
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from gpu_util import normalised_max_error, require_gpu

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent

# batch, n_q, n_k, d, type, mask, window, elements that pad a row; edges of the 32-row tiles, of two and four waves' turns at them
# (64 and 128 streamed rows), rows past the end in every wave, a wave without a tile, windows that begin in a later tile
FORMS = [(b, n_q, n_k, d, dtype, causal, window, pad)
         for d in (64, 128)
         for b, n_q, n_k, dtype, causal, window, pad in [
             (1, 1, 1, "bfloat16", False, None, 0), (2, 31, 33, "float16", False, None, 0), (3, 32, 32, "bfloat16", True, None, 8),
             (2, 65, 257, "bfloat16", False, None, 0), (1, 127, 95, "float16", False, None, 16), (5, 129, 129, "bfloat16", True, 40, 0),
             (2, 97, 640, "float16", "bottom_right", None, 0), (2, 300, 400, "bfloat16", "bottom_right", 200, 8),
             (1, 33, 1000, "bfloat16", "bottom_right", 17, 0), (1, 1030, 1030, "float16", True, None, 0), (4, 1000, 63, "bfloat16", False, None, 0)]]
# shapes whose default lies on either side of the lines of the rule, and what it picks for (forward, first backward, double-backward)
PICKS = [((16, 256, 64, True), (4, 4, 4)), ((33, 256, 64, False), (4, 2, 0)), ((33, 256, 64, True), (4, 2, 2)), ((64, 200, 128, False), (2, 0, 0)),
         ((2, 1024, 128, False), (4, 4, 4)), ((64, 128, 64, False), (4, 2, 2)), ((8, 1024, 128, True), (4, 4, 4)), ((8, 1024, 128, False), (4, 4, 0)),
         ((1, 4224, 128, False), (4, 4, 0)), ((256, 100, 64, True), (0, 0, 0))]

_CHILD = r"""
import sys, torch
sys.path[:0] = [{root!r} + "/flash-hob_amd"]
import fhog
out = []
def run(b, n_q, n_k, d, dtype, causal, window, pad, seed):
    g = torch.Generator().manual_seed(seed)
    def mk(n, s):
        t = torch.zeros(b, n, d + pad, dtype=getattr(torch, dtype), device="cuda")[..., :d]
        return t.copy_((torch.randn(b, n, d, generator=g) * s).to(t.dtype))
    q, do, ddq, k, v, ddk, ddv = mk(n_q, 1), mk(n_q, .1), mk(n_q, .1), mk(n_k, 1), mk(n_k, 1), mk(n_k, .1), mk(n_k, .1)
    scale = d ** -0.5
    o, L = fhog.attention_forward(q, k, v, scale, causal, window=window, use_hip=True)
    o2, L2 = fhog.attention_forward(q, k, v, scale, causal, window=window, use_hip=False)   # the same in every process
    o2 = mk(n_q, 0).copy_(o2)
    first = fhog.attention_backward(q, k, v, o2, do, L2, scale, causal, window=window, use_hip=True)
    second = fhog.flash_bwdbwd(q, k, v, o2, do, ddq, ddk, ddv, L2, scale, causal=causal, window=window, return_stats=True)
    out.append([t.cpu() for t in (o, L, *first, *second[:4], *second[4])])
for i, c in enumerate({cases!r}):
    run(*c, seed=i)
torch.save(out, sys.argv[1])
"""


def _run(path, tune, cases):
    r = subprocess.run([sys.executable, "-c", _CHILD.format(root=str(ROOT), cases=cases), str(path)],
                       env=dict(os.environ, FHOG_TUNE=tune), capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "ignored" not in r.stderr, r.stderr
    return torch.load(path, weights_only=True)


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


@pytest.mark.parametrize("waves", [4, 2])
def test_small_launches_agree_with_large_ones(tmp_path, waves):
    """Every form of call that the 16-bit kernels take. Same products of the same numbers: weights rounded to the type beside another
    running maximum (O), sums in another order, one rounding to the type: two units of it at the largest element. Row statistics stay
    fp32: 1e-5."""
    want = _run(tmp_path / "w", "small=0", FORMS)
    got = _run(tmp_path / "g", f"small={waves}", FORMS)
    names = ("o", "L", "dq", "dk", "dv", "dq2", "dk2", "dv2", "ddo", "d", "dd", "b")
    for form, a, b in zip(FORMS, got, want):
        if form[2] == 1:   # one key: P = 1 and dS = 0; what is left of dQ and dK is the rounding of d
            a, b = a[:2] + a[4:5], b[:2] + b[4:5]
        unit = 2.0 ** -7 if form[4] == "bfloat16" else 2.0 ** -10
        for name, x, y in zip(names, a, b):
            assert torch.isfinite(x.float()).all(), (form, name)
            assert normalised_max_error(x.float(), y.float()) <= (unit if x.dtype != torch.float32 else 1e-5), (form, name)


def test_rule_for_small_launches(tmp_path):
    """The bits of the default are those of the kernels that the rule is to pick."""
    cases = [(b, n, n, d, "bfloat16", causal, None, 0) for (b, n, d, causal), _ in PICKS]
    forced = {w: _run(tmp_path / f"w{w}", f"small={w}", cases) for w in (0, 2, 4)}
    default = _run(tmp_path / "d", "", cases)
    for i, (shape, picks) in enumerate(PICKS):
        for part, pick in zip((slice(0, 2), slice(2, 5), slice(5, None)), picks):
            assert all(torch.equal(x, y) for x, y in zip(default[i][part], forced[pick][i][part])), (shape, part)


# batch, n_q, n_k, mask, window: both sides of the lines at which the number of waves on the same rows changes, 63 to 65 groups of 128
# rows on the two sides together, 159 and 161 without a mask, 256 to 258 and 511 under a triangle
@pytest.mark.parametrize("shape", [(31, 100, 130, False, None), (32, 130, 100, True, 30), (53, 200, 128, False, None), (23, 385, 385, False, None),
                                   (64, 256, 256, True, None), (43, 300, 300, True, None), (73, 500, 300, False, None), (2, 90, 4000, "bottom_right", 100)])
@pytest.mark.parametrize("dtype,d", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 32), (torch.float16, 64)])
def test_passes_3_and_4_in_one_launch(shape, dtype, d):
    """The split-product sweeps for dQ2, ddO and dK2, dV2 side by side: bit for bit as from the passes launched one by one, and against
    the fp64 closed form at the gates of those sweeps."""
    from fhog import BwdBwdPlan
    from gpu_util import NAMES, errors, make_case, reference_fp64_cpu, with_caches
    batch, n_q, n_k, causal, window = shape
    if causal is True:
        n_k = n_q
    x = with_caches(make_case(batch, n_q, n_k, d, dtype, seed=81, grad_std=0.1), d ** -0.5, causal, window)
    plans = [BwdBwdPlan(x["Q"], x["K"], x["V"], x["O"], x["dO"], x["ddQ"], x["ddK"], x["ddV"], x["L"], d ** -0.5, causal=causal, window=window,
                        impl="fp32", schedule="fused_stats") for _ in range(2)]
    for p in plans:
        for t in p.outs:
            t.fill_(float("nan"))
    plans[0].run()
    for i in (5, 3, 4):
        plans[1].run(only_pass=i)
    torch.cuda.synchronize()
    for a, b in zip(plans[0].outs, plans[1].outs):
        assert torch.equal(a, b) and torch.isfinite(a.float()).all()
    sel = [0, batch // 2, batch - 1]
    ref = reference_fp64_cpu(x, d ** -0.5, causal, window, heads=sel)
    outs = dict(zip(("dq2", "dk2", "dv2", "ddo"), plans[0].outs))
    e = errors([outs[n].view(batch, -1, d)[sel] for n in NAMES], [ref[n] for n in NAMES])
    assert max(e.values()) < {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 2.5e-3}[dtype], e


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_weights_are_fp32_with_two_waves_on_the_same_rows(d, dtype):
    from test_gpu_split import test_weights_beside_16_bit_tensors_are_fp32 as check
    check(35, d, dtype)   # 70 groups of 128 rows a side


# both sides of the lines at which waves share rows and the two sweeps share a launch: 127 to 130 groups of 128 rows on both sides together,
# 159 and 161, 256 to 258 and 511 under a triangle, full rounds of 256 workgroups (whose sweeps run one after the other at d = 64 and 128)
@pytest.mark.parametrize("shape", [(64, 100, 127, False, None), (65, 33, 128, False, None), (43, 130, 200, False, None), (23, 385, 385, False, None),
                                   (128, 65, 40, True, None), (73, 300, 300, True, 70), (256, 33, 97, False, None), (8, 1030, 1030, True, None)])
@pytest.mark.parametrize("dtype,d", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 32), (torch.float16, 32)])
def test_first_backward_on_split_products(shape, dtype, d):
    """dQ beside dK and dV, whose sweep takes d = rowsum(O dO) itself, on padded rows, against fp64: the gates of the split products."""
    import fhog
    from gpu_util import make_case
    from oracle.bwdbwd_oracle import first_backward
    batch, n_q, n_k, causal, window = shape
    if causal is True:
        n_k = n_q
    x = make_case(batch, n_q, n_k, d, dtype, seed=82, grad_std=0.1)
    scale = d ** -0.5

    def padded(t):
        y = torch.full((*t.shape[:-1], d + 8), float("nan"), dtype=t.dtype, device=t.device)
        y[..., :d] = t
        return y[..., :d]

    o, L = fhog.attention_forward(x["Q"], x["K"], x["V"], scale, causal, window=window, use_hip=True)
    got = fhog.attention_backward(*map(padded, (x["Q"], x["K"], x["V"], o, x["dO"])), L, scale, causal, window=window, use_hip=True)
    sel = [0, batch // 2, batch - 1]
    c = {n: t[sel].double().cpu().numpy() for n, t in x.items()}
    want = first_backward(c["Q"], c["K"], c["V"], c["dO"], scale, causal, window)
    for name, g, w in zip(("dq", "dk", "dv"), got, want):
        assert torch.isfinite(g.float()).all()
        assert normalised_max_error(g[sel], w) < {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 2.5e-3}[dtype], name


# one side streams four times as many rows as the other and the two have more than 64 groups of 128 rows: each sweep runs by itself;
# and just inside of both lines
@pytest.mark.parametrize("shape", [(11, 40, 600, False, None), (11, 600, 40, False, None), (33, 130, 520, False, None), (33, 130, 519, False, None),
                                   (10, 40, 600, False, None), (40, 70, 300, "bottom_right", None), (9, 1000, 100, False, None)])
@pytest.mark.parametrize("dtype,d", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 32), (torch.float16, 32)])
def test_sweeps_of_lopsided_launches(shape, dtype, d):
    test_passes_3_and_4_in_one_launch(shape, dtype, d)
    test_first_backward_on_split_products(shape, dtype, d)
