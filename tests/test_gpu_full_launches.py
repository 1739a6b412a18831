"""GPU tier: launches that fill the GPU, where a workgroup's four waves have 32 rows each. fp32 tensors: the next tile is split behind the
MFMAs of this one (statistics sweeps and forward at d = 64), two workgroups share a CU (first order at d = 64, forward at d = 128). All: waves
whose rows lie past the end of their tensor compute nothing."""
import pytest
import torch

from gpu_util import NAMES, TOL, errors, make_case, reference_fp64_cpu, require_gpu, run_fhog, with_caches

pytestmark = pytest.mark.gpu

# slices, n_q, n_k, mask, window: one streamed row, the edges of the 32-row tiles, one tile to five, rows past the end in every wave, waves
# whose tiles are hidden while the others' are not, windows that begin in a later tile
FORMS = [(260, 33, 1, False, None), (260, 1, 31, False, None), (257, 130, 33, False, None), (260, 128, 64, False, None), (130, 257, 65, False, None),
         (520, 40, 40, True, None), (260, 160, 160, True, None), (200, 300, 300, True, 45), (520, 33, 150, "bottom_right", None), (200, 300, 420, "bottom_right", 70)]


def _slices(batch):
    """Those that are compared; every slice has to be finite."""
    return [0, 1, 7, 100, batch - 1]


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


def _first_order_fp64(x, scale, causal, window):
    """O and the gradients of Q, K, V of some slices in double precision, on materialised scores."""
    sel = _slices(x["Q"].shape[0])
    q, k, v = (x[n].double().cpu()[sel].requires_grad_(True) for n in ("Q", "K", "V"))
    s = q @ k.transpose(1, 2).contiguous() * scale
    i, j = torch.arange(q.shape[1])[:, None], torch.arange(k.shape[1])[None, :]
    i = i + (k.shape[1] - q.shape[1] if causal == "bottom_right" else 0)
    hidden = (j > i) if causal else torch.zeros_like(j > i)
    if window is not None:
        hidden = hidden | (i - j >= window)
    o = torch.softmax(s.masked_fill(hidden, float("-inf")), -1) @ v
    return (o.detach(), *torch.autograd.grad(o, (q, k, v), x["dO"].double().cpu()[sel]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("form", FORMS, ids=str)
def test_first_order_and_double_backward(form, d, dtype):
    """The gate of the type. One key: dS is rounding of d, and so are dQ, dK, dQ2 and dK2."""
    import fhog
    batch, n_q, n_k, causal, window = form
    x = make_case(batch, n_q, n_k, d, dtype, seed=n_q + n_k)
    scale, sel = d ** -0.5, _slices(batch)
    leaves = [x[n].clone().requires_grad_(True) for n in ("Q", "K", "V")]
    out = fhog.attention(*(t[None] for t in leaves), causal, window)[0]
    got = (out.detach(), *torch.autograd.grad(out, leaves, x["dO"]))
    for name, g, r in zip(("o", "dq", "dk", "dv"), got, _first_order_fp64(x, scale, causal, window)):
        assert torch.isfinite(g).all(), name
        if n_k > 1 or name in ("o", "dv"):
            assert (g.double().cpu()[sel] - r).abs().max() <= TOL[dtype] * r.abs().max(), name
    c = with_caches(x, scale, causal, window)
    outs = run_fhog(c, scale, causal, window=window)
    ref = reference_fp64_cpu({n: t for n, t in x.items()}, scale, causal, window, heads=sel)
    for name, e in errors([t.cpu()[sel] for t in outs], [torch.from_numpy(ref[n]) for n in NAMES]).items():
        if n_k > 1 or name in ("dv2", "ddo"):
            assert e <= TOL[dtype], (name, e)
    assert all(torch.isfinite(t).all() for t in outs)
