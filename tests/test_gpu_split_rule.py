"""GPU tier: how many splits passes 3 and 4 run with at d = 128 (rounds of workgroups under the mask against the cost of
combining): whatever the rule picks, results are those of the launch that does not split. The picks themselves are in
tests/test_launch_rules_host.py, launches whose picks are known in tests/test_gpu_large_kernels.py."""
import pytest
import torch

from gpu_util import NAMES, make_case, normalised_max_error, require_gpu, run_fhog, with_caches

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


# keys without a query at the front of the K side (statistics sweep split), a small launch, uneven work of a causal mask, window, 1 | 8 splits, none
@pytest.mark.parametrize("shape", [(16, 1000, 3001, "bottom_right", 700), (1, 300, 5000, "bottom_right", 64), (2, 2048, 2048, True, None),
                                   (24, 1536, 1536, True, 100), (3, 4095, 513, False, None), (40, 1025, 1024, False, None)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_by_rounds(shape, dtype):
    batch, n_q, n_k, causal, window = shape
    scale = 128 ** -0.5
    x = with_caches(make_case(batch, n_q, n_k, 128, dtype, seed=72, grad_std=0.1), scale, causal, window)
    split, whole = [run_fhog(x, scale, causal, window=window, split=s) for s in (True, False)]
    # sums in another order, rounded once: one unit of the type at the largest element (2^-8 for bf16, 2^-11 for fp16)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for name, a, b in zip(NAMES, split, whole):
        assert normalised_max_error(a, b.float()) <= unit, name


@pytest.mark.parametrize("schedule", ["three_sweep", "ddo_early"])
@pytest.mark.parametrize("shape", [(4, 4096, 4096, True, 128), (16, 1000, 3001, "bottom_right", 40)])
def test_schedules_run_as_asked_where_pass_3_does_not_split(shape, schedule):
    """Few enough workgroups that passes may split, and a mask under which pass 3 keeps one workgroup per tile: the schedule asked for
    runs, with the bits of the call that has no workspace for splits."""
    batch, n_q, n_k, causal, window = shape
    scale = 128 ** -0.5
    x = with_caches(make_case(batch, n_q, n_k, 128, torch.bfloat16, seed=77, grad_std=0.1), scale, causal, window)
    got, want = (run_fhog(x, scale, causal, window=window, schedule=schedule, split=s) for s in (True, False))
    other = run_fhog(x, scale, causal, window=window, schedule="fused_stats" if schedule == "three_sweep" else "four_pass")
    assert any(not torch.equal(a, b) for a, b in zip(got, other))
    if schedule == "three_sweep":   # its sweeps have no split form
        assert bool(torch.equal(got[0], want[0])) and bool(torch.equal(got[3], want[3]))
    # the sweep for dd of the other one, and pass 4, may have split: sums in another order, one unit of the type
    for name, a, b in zip(NAMES, got, want):
        assert normalised_max_error(a, b.float()) <= 2.0 ** -8, name
