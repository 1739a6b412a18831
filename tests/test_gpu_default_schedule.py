"""GPU tier: what the entry points run when no schedule is asked for."""
import pytest
import torch

from gpu_util import NAMES, make_case, normalised_max_error, require_gpu, run_fhog, with_caches

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


@pytest.mark.parametrize("case", [(torch.bfloat16, 3, 333, 333, 128, True), (torch.float16, 2, 100, 777, 64, False),
                                  (torch.bfloat16, 1, 2048, 2048, 64, True), (torch.bfloat16, 70, 512, 512, 128, True),
                                  (torch.float32, 2, 96, 160, 64, False)])
def test_default_is_the_fused_statistics_schedule(case):
    """Bit for bit the schedule asked for by name, and the four sweeps' statistics up to fp32 summation order (the bound of
    the test of that sweep alone, 1e-3; the outputs are then rounded to 16 bits: one unit in the last place, 2^-8)."""
    dtype, batch, n_q, n_k, d, causal = case
    x = with_caches(make_case(batch, n_q, n_k, d, dtype, seed=62, grad_std=0.1), d ** -0.5, causal)
    base = run_fhog(x, d ** -0.5, causal, return_stats=True)
    named = run_fhog(x, d ** -0.5, causal, schedule="fused_stats", return_stats=True)
    four = run_fhog(x, d ** -0.5, causal, schedule="four_pass", return_stats=True)
    for a, b in zip((*base[:4], *base[4]), (*named[:4], *named[4])):
        assert torch.equal(a, b)
    for name, a, b in zip(NAMES, base[:4], four[:4]):
        assert normalised_max_error(a, b.float()) < (1e-5 if dtype == torch.float32 else 2 ** -8), name
    for name, a, b in zip(("d", "dd", "b"), base[4], four[4]):
        assert normalised_max_error(a, b) < 1e-3, name
