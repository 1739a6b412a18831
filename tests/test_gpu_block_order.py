"""GPU tier: the order in which workgroups take the tiles of a masked launch (decode_block), around the 32nd, 64th and 65th
workgroup of an XCD: every tile of every slice is computed, exactly as in a launch of another number of slices."""
import pytest
import torch

from gpu_util import TOL, make_case, require_gpu, run_fhog

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


# slices per XCD (a multiple of 8 slices, slices / 8 each) x tiles of 128 rows: 32, 33, 63, 64 and 65 workgroups of an XCD
@pytest.mark.parametrize("slices,tiles", [(64, 4), (24, 11), (168, 3), (128, 4), (40, 13)])
@pytest.mark.parametrize("d,causal", [(32, True), (64, True), (64, "bottom_right"), (128, True)])
def test_batched_launch_equals_its_slices(slices, tiles, d, causal):
    import fhog
    n = 128 * tiles - 5
    scale = d ** -0.5
    x = make_case(slices, n, n if causal is True else n + 70, d, torch.bfloat16, seed=71, grad_std=0.1)

    def outputs(x):
        o, L = fhog.attention_forward(x["Q"], x["K"], x["V"], scale, causal, use_hip=True)
        first = fhog.attention_backward(x["Q"], x["K"], x["V"], o, x["dO"], L, scale, causal, use_hip=True)
        second = [t for s in ("fused_stats", "three_sweep") for t in run_fhog(dict(x, O=o, L=L), scale, causal, schedule=s, split=False)]
        return (o, L, *first, *second)

    got = outputs(x)
    # Copies of one slice, enough that both launches lie on the same side of every line at which the number of workgroups changes the
    # order of sums: the highest is 256, up to which the statistics sweep of the split products puts four waves on the same rows.
    copies = 256 // tiles + 8
    assert min(copies, slices) * tiles >= 256
    for s in (0, slices // 2, slices - 1):
        other = outputs({name: t[s:s + 1].expand(copies, -1, -1).contiguous() for name, t in x.items()})
        for a, b in zip(got, other):
            assert torch.equal(a[s], b[0]) and torch.equal(a[s], b[-1])
    assert all(torch.isfinite(t.float()).all() for t in got)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_two_sweeps_in_turn_equal_one_after_the_other(dtype):
    """Split products at d = 32: 512 workgroups of 128 rows a side take turns with those of the other side, 1040 do not. The first backward of 16-bit tensors
    has two launches by then, whose dK, dV take the row sums d from the sweep for dQ instead of adding them up in another order: fp32 ones only."""
    import fhog
    slices, copies, n, scale = 64, 130, 1019, 32 ** -0.5
    x = make_case(slices, n, n, 32, dtype, seed=73, grad_std=0.1)

    def outputs(x):
        o, L = fhog.attention_forward(x["Q"], x["K"], x["V"], scale, True, use_hip=True)
        first = fhog.attention_backward(x["Q"], x["K"], x["V"], o, x["dO"], L, scale, True, use_hip=True) if dtype == torch.float32 else ()
        return (*first, *run_fhog(dict(x, O=o, L=L), scale, True))

    got = outputs(x)
    assert all(torch.isfinite(t.float()).all() for t in got)
    for s in (0, slices // 2, slices - 1):
        other = outputs({name: t[s:s + 1].expand(copies, -1, -1).contiguous() for name, t in x.items()})
        assert all(torch.equal(a[s], b[0]) and torch.equal(a[s], b[-1]) for a, b in zip(got, other))


# fp32 tensors: launches whose workgroups have a CU to themselves, share it with another, take turns by sweep or share it with two more, each against copies
# of a slice in a launch of another of these kinds, with the two sweeps in one launch in both
@pytest.mark.parametrize("slices,copies,n_q,n_k,d,causal,window", [(24, 40, 1100, 1100, 64, True, None), (16, 30, 1000, 1700, 64, "bottom_right", 600),
                                                                   (18, 40, 900, 1300, 64, "bottom_right", 500), (30, 45, 1019, 1000, 32, False, None)])
def test_company_does_not_change_the_first_backward(slices, copies, n_q, n_k, d, causal, window):
    import fhog
    scale = d ** -0.5
    x = make_case(slices, n_q, n_k, d, torch.float32, seed=75)

    def outputs(x):
        o, L = fhog.attention_forward(x["Q"], x["K"], x["V"], scale, causal, window=window, use_hip=True)
        return fhog.attention_backward(x["Q"], x["K"], x["V"], o, x["dO"], L, scale, causal, window=window, use_hip=True)

    got = outputs(x)
    for s in (0, slices // 2, slices - 1):
        other = outputs({name: t[s:s + 1].expand(copies, -1, -1).contiguous() for name, t in x.items()})
        assert all(torch.equal(a[s], b[0]) and torch.equal(a[s], b[-1]) for a, b in zip(got, other))
    q, k, v = (x[name][-1].double().cpu().requires_grad_(True) for name in ("Q", "K", "V"))
    i, j = torch.arange(n_q)[:, None] + (n_k - n_q if causal == "bottom_right" else 0), torch.arange(n_k)[None, :]
    hidden = ((j > i) | (i - j >= (window or n_k))) if causal else torch.zeros(n_q, n_k, dtype=torch.bool)
    o = torch.softmax((q @ k.T * scale).masked_fill(hidden, float("-inf")), -1) @ v
    for a, r in zip(got, torch.autograd.grad(o, (q, k, v), x["dO"][-1].double().cpu())):
        assert (a[-1].double().cpu() - r).abs().max() <= TOL[torch.float32] * r.abs().max()
