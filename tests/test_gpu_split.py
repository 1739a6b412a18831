"""GPU tier: the split-product kernels (fp32-accurate contractions on the 16-bit matrix instructions)."""
import pytest
import torch

from gpu_util import NAMES, errors, make_case, normalised_max_error, reference_fp64_cpu, require_gpu, run_fhog, with_caches
from oracle.bwdbwd_oracle import first_backward, forward_o_lse

pytestmark = pytest.mark.gpu
# fp32: the gate of the fp32 family. 16-bit tensors: products and sums are as accurate, but O is rounded before
# d = rowsum(O * dO) and every result is rounded once; the fp16 gate is the bf16 one times the ratio of the units, 2^-3.
TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2, torch.float16: 2.5e-3}


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


@pytest.mark.parametrize("dtype", list(TOL))
@pytest.mark.parametrize("d", [32, 64, 128])
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


@pytest.mark.parametrize("case", [(t, d) for t in TOL for d in (32, 64, 128) if t == torch.float32 or d == 32])
@pytest.mark.parametrize("shape", [(1, 1, 1, False, None), (1, 33, 65, False, None), (3, 64, 300, "bottom_right", 40),
                                   (1, 97, 97, True, 1), (70, 128, 95, False, None), (130, 161, 161, True, 33),
                                   (130, 128, 130, "bottom_right", None)])
def test_first_order_on_split_products(shape, case):
    """Forward and first backward in every wave split, ragged on both sides, rows whose window starts in a later tile."""
    import fhog
    dtype, d = case
    batch, n_q, n_k, causal, window = shape
    x = make_case(batch, n_q, n_k, d, dtype, seed=64)
    scale = d ** -0.5
    o, L = fhog.attention_forward(x["Q"], x["K"], x["V"], scale, causal, window=window, use_hip=True)
    got = fhog.attention_backward(x["Q"], x["K"], x["V"], o, x["dO"], L, scale, causal, window=window, use_hip=True)
    sel = slice(None) if batch < 4 else slice(0, batch, 43)
    c = {n: t[sel].double().cpu().numpy() for n, t in x.items()}
    o_ref, l_ref = forward_o_lse(c["Q"], c["K"], c["V"], scale, causal, window)
    assert normalised_max_error(o[sel], o_ref) < (1e-4 if dtype == torch.float32 else TOL[dtype] / 2)   # rounded once
    assert (L[sel].double().cpu() - torch.from_numpy(l_ref)).abs().max() < 1e-4
    want = first_backward(c["Q"], c["K"], c["V"], c["dO"], scale, causal, window)
    for name, g, w in zip(("dq", "dk", "dv"), got, want):
        # one visible key per query (n_k = 1 or a window of 1): dS vanishes identically and the rounding of O is what is left
        floor = 1e-4 if dtype == torch.float32 else 1e-2
        assert (g[sel].double().cpu() - torch.from_numpy(w)).abs().max() < TOL[dtype] * abs(w).max() + floor, name


@pytest.mark.parametrize("dtype", list(TOL))
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("shape", [(1, 33, 66, False, None), (2, 40, 333, False, None), (1, 290, 290, True, None), (1, 31, 400, "bottom_right", 200)])
def test_statistics_sweep_that_stages_nothing(shape, d, dtype):
    """Four waves on the same rows reading their own tiles: three tiles for four waves, eleven (a remainder in the last round and
    in the last tile), a causal range that grows, a band whose first tile is not the first one. Padded rows on the streamed side. With 16-bit tensors O is rounded before
    d = rowsum(O * dO): an absolute error up to 2^-9 sum |O dO|, which the largest |d| of some 30 rows is well above; the d of a
    single row need not be."""
    from fhog import BwdBwdPlan
    batch, n_q, n_k, causal, window = shape
    x = with_caches(make_case(batch, n_q, n_k, d, dtype, seed=67), d ** -0.5, causal, window)
    ref = reference_fp64_cpu(x, d ** -0.5, causal, window)

    def padded(t):
        y = torch.full((*t.shape[:-1], d + 8), float("nan"), dtype=t.dtype, device=t.device)
        y[..., :d] = t
        return y[..., :d]

    for lay in (lambda t: t, padded):
        plan = BwdBwdPlan(x["Q"], lay(x["K"]), lay(x["V"]), x["O"], x["dO"], x["ddQ"], lay(x["ddK"]), lay(x["ddV"]), x["L"], d ** -0.5,
                          causal=causal, window=window, impl="fp32")
        for passes in ((5,), (1, 2)):
            plan.ws.fill_(float("nan"))
            for i in passes:
                plan.run(only_pass=i)
            torch.cuda.synchronize()
            for got, name in zip(plan.ws[:3 * batch * n_q].view(3, -1), ("d", "dd", "b")):
                want = torch.as_tensor(ref[name]).reshape(-1)
                assert normalised_max_error(got, want) < (1e-4 if dtype == torch.float32 else 5e-3), (name, passes)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("batch", [2, 70, 140])
def test_weights_beside_16_bit_tensors_are_fp32(batch, d, dtype):
    """Sums of the weights against +-pairs cancel down to their spread, 2^-13 of a weight here: what is left of them shows how many
    bits the weights carried. With fp32 ones the roundings of the exponent and of L remain, 2^-22 of a weight each at fewer than 256
    keys: 2^-8 of the result, besides its own rounding to the type (16 bits of a weight leave 2^-6). Four, two and one wave on the
    same rows."""
    import fhog
    n, s = 190, 2.0 ** -6.5
    g = torch.Generator().manual_seed(73)
    q, k = ((torch.randn(batch, n, d, generator=g) * s).to(dtype).cuda() for _ in range(2))
    pairs = torch.randn(batch, n, d, generator=g).to(dtype).cuda()
    pairs[:, 1::2] = -pairs[:, ::2]
    zero = torch.zeros_like(q)
    scale = d ** -0.5
    sel = slice(0, batch, 43)
    p = torch.softmax(q[sel].double().cpu() @ k[sel].double().cpu().transpose(1, 2).contiguous() * scale, -1)
    x = pairs[sel].double().cpu()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    o, L = fhog.attention_forward(q, k, pairs, scale)
    got = {"ddo": (fhog.flash_bwdbwd(q, k, zero, o, zero, zero, zero, pairs, L, scale, impl="fp32")[3], p @ x)}
    if d == 32:   # the first-order kernels of the other head dims are 16-bit ones
        got["o"] = (o, p @ x)
        got["dv"] = (fhog.attention_backward(q, k, zero, zero, pairs, L, scale, False)[2], p.transpose(1, 2).contiguous() @ x)
    for name, (a, want) in got.items():
        e = normalised_max_error(a[sel], want)
        assert e < unit + 2.0 ** -8, (name, e)


@pytest.mark.parametrize("dtype,d,value", [(t, d, x) for x in (float("inf"), float("-inf"), float("nan"), 3.4e38)
                                           for t, d in ((torch.float32, 32), (torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 32),
                                                        (torch.float16, 32)) if t == torch.float32 or x != 3.4e38])
@pytest.mark.parametrize("batch", [2, 70, 140])
def test_numbers_that_bf16_cannot_hold(batch, dtype, d, value):
    """One infinity, NaN or number beyond bf16's largest in V, dO or ddV changes its own column of O, dV and ddO alone: infinite with
    its sign, the weighted sum where the number is finite (fp32 tensors; beside 16-bit ones the three terms of a weight may meet an
    infinity with both signs, so not finite is all that is said). One in a row of K, where an infinite score hides the key or takes
    the row, stays in the rows that it takes."""
    import fhog
    n, row, col = 190, 67, 5
    g = torch.Generator().manual_seed(76)
    q, k, v, do, ddv = (torch.randn(batch, n, d, generator=g).to(dtype).cuda() for _ in range(5))
    zero = torch.zeros_like(q)
    scale = d ** -0.5

    def marked(t):
        t = t.clone()
        t[:, row, col] = value
        return t

    def others(t):
        return torch.cat([t[..., :col], t[..., col + 1:]], -1)

    o, L = fhog.attention_forward(q, k, v, scale, use_hip=True)
    o1, L1 = fhog.attention_forward(q, k, marked(v), scale, use_hip=True)
    p = torch.softmax(q.double().cpu() @ k.double().cpu().transpose(1, 2).contiguous() * scale, -1)
    second = lambda x: fhog.flash_bwdbwd(q, k, zero, zero, zero, zero, zero, x, L, scale)[3]
    dv = lambda x: fhog.attention_backward(q, k, zero, zero, x, L, scale, False, use_hip=True)[2]
    assert torch.equal(L, L1)
    for got, plain, weight in ((o1, o, p[:, :, row]), (second(marked(ddv)), second(ddv), p[:, :, row]),
                               (dv(marked(do)), dv(do), p[:, row, :])):
        assert torch.equal(others(got), others(plain))
        x = got[..., col].double().cpu()
        if dtype != torch.float32:
            assert not torch.isfinite(x).any()
        elif value == 3.4e38:   # the marked element decides the sum; fp32 roundings of the exponent and of L, 2^-22 of a weight each at scores below 16
            assert (x / (weight * 3.4e38) - 1).abs().max() < 1e-5
        elif value != value:
            assert torch.isnan(x).all()
        else:
            assert (x == value).all()
    # a score of -Inf hides its key, one of +Inf or NaN takes the row
    if dtype == torch.float32 and abs(value) == float("inf"):
        o2 = fhog.attention_forward(q, marked(k), v, scale, use_hip=True)[0]
        hidden = q[..., col] * value < 0
        keys = [j for j in range(n) if j != row]
        want = fhog.attention_forward(q, k[:, keys].contiguous(), v[:, keys].contiguous(), scale, use_hip=True)[0]
        assert normalised_max_error(o2[hidden], want[hidden]) < 1e-5 and torch.isnan(o2[~hidden]).all()
