"""GPU tier: double-backwards of fp32 tensors with one output to a workgroup (fhog_split_few.hip). FHOG_TUNE chooses between them and the kernels
with both outputs of a side in a workgroup, in one process each."""
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from gpu_util import NAMES, errors, require_gpu
from oracle.bwdbwd_oracle import closed_form

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent

# batch, n_q, n_k, d, mask, window, elements that pad a row: edges of the 32-row tiles and of two and four waves' turns at them (64 and 128
# streamed rows), rows past the end in every wave, waves without a tile, windows that begin in a later tile, slices dealt out over the XCDs
FORMS = [(b, n_q, n_k, d, causal, window, pad)
         for d in (32, 64, 128)
         for b, n_q, n_k, causal, window, pad in [
             (1, 1, 1, False, None, 0), (2, 31, 33, False, None, 4), (3, 32, 32, True, None, 0), (2, 65, 257, False, None, 0),
             (1, 129, 95, False, None, 8),
             (5, 129, 129, True, 40, 0), (2, 97, 640, "bottom_right", None, 0), (2, 300, 400, "bottom_right", 200, 4), (1, 33, 1000, "bottom_right", 17, 0),
             (9, 70, 64, False, None, 0), (1, 515, 515, True, None, 0)]]
# both sides of the lines of the rule, and whether it takes them
PICKS = [((8, 256, 256, 32, False), 1), ((12, 256, 256, 32, False), 0), ((8, 512, 512, 64, False), 1), ((16, 256, 256, 64, False), 0), ((16, 512, 512, 64, False), 0),
         ((5, 955, 955, 128, True), 1), ((16, 256, 256, 128, False), 1), ((32, 256, 256, 128, False), 0), ((8, 48, 2858, 128, False), 1)]

_CHILD = r"""
import sys, torch
sys.path[:0] = [{root!r} + "/flash-hob_amd"]
import fhog
out = []
def run(b, n_q, n_k, d, causal, window, pad, seed):
    g = torch.Generator().manual_seed(seed)
    def mk(n, s):
        t = torch.zeros(b, n, d + pad, device="cuda")[..., :d]
        return t.copy_(torch.randn(b, n, d, generator=g) * s)
    q, do, ddq, k, v, ddk, ddv = mk(n_q, 1), mk(n_q, 1), mk(n_q, 1), mk(n_k, 1), mk(n_k, 1), mk(n_k, 1), mk(n_k, 1)
    o, L = fhog.attention_forward(q, k, v, d ** -0.5, causal, window=window, use_hip=False)
    o = mk(n_q, 0).copy_(o)
    outs = fhog.flash_bwdbwd(q, k, v, o, do, ddq, ddk, ddv, L, d ** -0.5, causal=causal, window=window)
    out.append([t.cpu() for t in (*outs, q, k, v, do, ddq, ddk, ddv)])
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


@pytest.mark.parametrize("few", [0, 1])
def test_every_form_against_the_closed_form(tmp_path, few):
    """Either kernels on every form of call, at the gate of fp32 tensors. One key: dS is rounding of d, and so are dQ2, dK2."""
    for form, (*outs, q, k, v, do, ddq, ddk, ddv) in zip(FORMS, _run(tmp_path / "o", f"few={few}", FORMS)):
        d, causal, window = form[3:6]
        ref = closed_form(*(t.double().numpy() for t in (q, k, v, do, ddq, ddk, ddv)), d ** -0.5, causal, window=window)
        err = errors(outs, [torch.from_numpy(ref[n]) for n in NAMES])
        assert all(torch.isfinite(t).all() for t in outs), form
        for name, e in err.items():
            if form[2] > 1 or name in ("dv2", "ddo"):
                assert e <= 1e-4, (form, name, e)


def test_rule(tmp_path):
    """The bits of the default are those of the kernels that the rule is to pick."""
    cases = [(*shape, None, 0) for shape, _ in PICKS]
    forced = [_run(tmp_path / f"f{w}", f"few={w}", cases) for w in (0, 1)]
    for i, ((shape, pick), got) in enumerate(zip(PICKS, _run(tmp_path / "d", "", cases))):
        if shape[3] > 32:   # four waves add up in the same order there, whichever kernels run: test_launch_rules_host.py has that line
            assert any(not torch.equal(x, y) for x, y in zip(forced[0][i][:4], forced[1][i][:4])), shape
        assert all(torch.equal(x, y) for x, y in zip(got[:4], forced[pick][i][:4])), shape
