"""GPU tier: the 16-bit kernels with 128 rows to a workgroup, split launches and the passes of the opt-in schedules on launches that the kernels for
small launches (fhog_small.hip) take by default. FHOG_TUNE=small=0 keeps them out, in one process for all cases."""
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from gpu_util import normalised_max_error, reference_fp64_cpu, require_gpu

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent
ORDER = ("dq2", "dk2", "dv2", "ddo")   # a plan's outputs

# batch, n_q, n_k, d, type, mask, window, row padding, splits of passes 3 and 4 in the launch that they share (one side, both, unequal ones; ragged ends)
SPLITS = [(1, 2048, 2048, 64, "bfloat16", False, None, 0, (8, 8)), (1, 2048, 2048, 64, "float16", True, None, 8, (8, 8)),
          (2, 1000, 1500, 64, "bfloat16", "bottom_right", None, 0, (4, 4)), (1, 1536, 1536, 64, "bfloat16", True, 300, 0, (4, 4)),
          (1, 130, 4100, 64, "bfloat16", False, None, 0, (16, 1)), (2, 2600, 700, 64, "float16", False, None, 64, (2, 8)),
          (1, 1030, 3100, 64, "bfloat16", "bottom_right", None, 0, (8, 4)), (2, 2050, 1030, 64, "bfloat16", False, None, 0, (2, 4)),
          (1, 2048, 2048, 128, "bfloat16", True, None, 0, (8, 8)), (2, 1000, 1500, 128, "float16", False, None, 0, (4, 4)),
          (1, 1536, 1536, 128, "bfloat16", "bottom_right", 700, 0, (4, 4)), (1, 2000, 1024, 128, "bfloat16", False, None, 8, (2, 4)),
          (3, 1030, 2050, 128, "float16", False, None, 0, (4, 2)), (2, 520, 2300, 128, "bfloat16", "bottom_right", None, 0, (8, 2)),
          (3, 4095, 513, 128, "bfloat16", False, None, 0, (1, 8))]
# ragged lengths, one row, fewer keys than queries, band masks, padded rows, both types
FORMS = [(b, n_q, n_k, d, dtype, causal, window, pad, None)
         for d in (64, 128)
         for b, n_q, n_k, dtype, causal, window, pad in [
             (1, 1, 1, "bfloat16", False, None, 0), (2, 31, 33, "float16", False, None, 0), (3, 100, 77, "bfloat16", False, None, 0), (2, 33, 129, "bfloat16", False, None, 8),
             (9, 384, 128, "float16", False, None, 0), (2, 333, 333, "bfloat16", True, None, 0), (5, 257, 257, "float16", True, 65, 0),
             (3, 200, 456, "bfloat16", "bottom_right", None, 0), (3, 300, 400, "float16", "bottom_right", 200, 16), (3, 96, 160, "bfloat16", "bottom_right", 1, 0)]]

_CHILD = r"""
import sys, torch
sys.path[:0] = [{root!r} + "/flash-hob_amd", {root!r}, {root!r} + "/tests"]
from fhog import BwdBwdPlan
from gpu_util import make_case, with_caches

def padded(t, pad):
    wide = torch.zeros(*t.shape[:-1], t.shape[-1] + pad, dtype=t.dtype, device=t.device)
    wide[..., :t.shape[-1]] = t
    return wide[..., :t.shape[-1]]

def run(case, schedule, split, passes=None):
    b, n_q, n_k, d, dtype, causal, window, pad, _ = case
    p = BwdBwdPlan(*(x[n] for n in ("Q", "K", "V", "O", "dO", "ddQ", "ddK", "ddV", "L")), d ** -0.5, causal=causal, window=window, impl="bf16",
                   schedule=schedule, split=split)
    p.ws_all.fill_(float("nan"))
    for t in p.outs:
        t.fill_(float("nan"))
    if passes is None:
        p.run()
    for i in passes or ():
        p.run(only_pass=i)
    torch.cuda.synchronize()
    written = (~torch.isnan(p.ws_all.view(-1))).nonzero()[-1].item() + 1
    return dict(outs=[t.cpu() for t in p.outs], stats=[t.cpu() for t in p.ws.view(3, b, n_q)], written=written)

out = []
for i, (case, schedules) in enumerate({cases!r}):
    b, n_q, n_k, d, dtype, causal, window, pad, _ = case
    print(i, case, flush=True)
    x = with_caches(make_case(b, n_q, n_k, d, getattr(torch, dtype), seed=900 + i, grad_std=0.1), d ** -0.5, causal, window)
    x = {{n: padded(t, pad) if n != "L" else t for n, t in x.items()}}
    res = dict(x={{n: t.cpu() for n, t in x.items()}})
    for s in schedules:
        res[s, "whole"] = run(case, s, False)
        if case[-1]:
            res[s, "split"] = run(case, s, True)
        else:
            res[s, "passes"] = run(case, s, False, passes=dict(ddo_early=(1, 6, 7, 4), three_sweep=(8, 7, 4))[s])
    out.append(res)
torch.save(out, sys.argv[1])
"""


def _run(path, cases):
    r = subprocess.run([sys.executable, "-c", _CHILD.format(root=str(ROOT), cases=cases), str(path)], env=dict(os.environ, FHOG_TUNE="small=0"),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-2000:]
    assert "ignored" not in r.stderr, r.stderr
    return torch.load(path, weights_only=True)


@pytest.fixture(scope="module")
def runs(tmp_path_factory):
    require_gpu()
    cases = [(c, ("fused_stats", "four_pass")) for c in SPLITS] + [(c, ("ddo_early", "three_sweep")) for c in FORMS]
    return _run(tmp_path_factory.mktemp("large") / "out", cases)


def _reference(case, x):
    return reference_fp64_cpu(x, case[3] ** -0.5, case[5], window=case[6])


@pytest.mark.parametrize("i", range(len(SPLITS)))
def test_split_launches(runs, i):
    """The gates of the split launches (tests/test_gpu_parity.py): outputs against the fp64 closed form, row statistics equal to the launch that does not
    split up to summation order, outputs within a rounding of it. How far the workspace was written tells the splits that ran."""
    case, r = SPLITS[i], runs[i]
    b, n_q, n_k, d = case[:4]
    x, y = case[8]
    ref = _reference(case, r["x"])
    for s in ("fused_stats", "four_pass"):
        split, whole = r[s, "split"], r[s, "whole"]
        stats = (3 * b * n_q + 3) // 4 * 4
        assert split["written"] == stats + 2 * d * b * ((x * n_q if x > 1 else 0) + (y * n_k if y > 1 else 0)), (s, split["written"])
        assert whole["written"] == 3 * b * n_q
        for res in (split, whole):
            assert max(normalised_max_error(o.view(b, -1, d), ref[n]) for n, o in zip(ORDER, res["outs"])) < 2e-2, s
            assert max(normalised_max_error(t, ref[n]) for n, t in zip(("d", "dd", "b"), res["stats"])) < 1e-2, s
        for t, u in zip(split["stats"], whole["stats"]):
            assert normalised_max_error(t, u) < 1e-5, s
        for t, u in zip(split["outs"], whole["outs"]):
            assert normalised_max_error(t, u.float()) < 1e-2, s


@pytest.mark.parametrize("schedule", ["ddo_early", "three_sweep"])
@pytest.mark.parametrize("i", range(len(FORMS)))
def test_schedules_run_their_own_passes(runs, i, schedule):
    """Bit for bit passes 1, 6, 7, 4 and 8, 7, 4 run one by one, and the gates of tests/test_gpu_schedules.py against the fp64 closed form."""
    case, r = FORMS[i], runs[len(SPLITS) + i]
    b, d = case[0], case[3]
    whole, passes = r[schedule, "whole"], r[schedule, "passes"]
    for t, u in zip(whole["outs"] + whole["stats"], passes["outs"] + passes["stats"]):
        assert torch.equal(t, u) and torch.isfinite(t.float()).all()
    ref = _reference(case, r["x"])
    assert max(normalised_max_error(o.view(b, -1, d), ref[n]) for n, o in zip(ORDER, whole["outs"])) < 2e-2
    assert max(normalised_max_error(t, ref[n]) for n, t in zip(("d", "dd", "b"), whole["stats"])) < 1e-2
