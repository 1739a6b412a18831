"""GPU tier: the split-product kernels (fp32-accurate contractions on the 16-bit matrix instructions) at d = 32 and 64."""
import pytest
import torch

from gpu_util import NAMES, errors, make_case, normalised_max_error, reference_fp64_cpu, require_gpu, run_fhog, with_caches

pytestmark = pytest.mark.gpu
# fp32: the gate of the fp32 family. 16-bit tensors: products and sums are as accurate, but O is rounded before
# d = rowsum(O * dO) and every result is rounded once; the fp16 gate is the bf16 one times the ratio of the units, 2^-3.
TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 2.5e-3}


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


@pytest.mark.parametrize("dtype", list(TOL))
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("shape", [(1, 1, 1, False, None), (1, 33, 65, False, None), (3, 64, 300, "bottom_right", 40),
                                   (1, 97, 97, True, 1), (70, 128, 95, False, None), (130, 161, 161, True, 33),
                                   (130, 128, 130, "bottom_right", None)])
def test_double_backward_on_split_products(shape, d, dtype):
    """Every wave split (4, 2 or 1 waves on the same rows), ragged tiles on both sides, masks and windows; the statistics of the
    fused sweep against those of the separate ones."""
    from fhog import BwdBwdPlan
    batch, n_q, n_k, causal, window = shape
    x = with_caches(make_case(batch, n_q, n_k, d, dtype, seed=63), d ** -0.5, causal, window)
    outs = run_fhog(x, d ** -0.5, causal, window=window, impl="fp32", return_stats=True)
    ref = reference_fp64_cpu(x, d ** -0.5, causal, window)
    e = errors(outs[:4], [ref[n] for n in NAMES])
    assert max(e.values()) < TOL[dtype], e
    for got, name in zip(outs[4], ("d", "dd", "b")):
        assert normalised_max_error(got, ref[name]) < (1e-4 if dtype == torch.float32 else 5e-3), name
    plan = BwdBwdPlan(x["Q"], x["K"], x["V"], x["O"], x["dO"], x["ddQ"], x["ddK"], x["ddV"], x["L"], d ** -0.5,
                      causal=causal, window=window, impl="fp32")
    plan.ws.fill_(float("nan"))
    for i in (1, 2):
        plan.run(only_pass=i)
    torch.cuda.synchronize()
    for got, fused, name in zip(plan.ws.view(3, -1), outs[4], ("d", "dd", "b")):
        assert normalised_max_error(got, fused.reshape(-1)) < 1e-4, name
