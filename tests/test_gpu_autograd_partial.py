"""GPU tier: autograd chains in which a node receives no gradient for some of its outputs."""
import itertools

import pytest
import torch

from gpu_util import normalised_max_error, require_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


def _torch_attention(q, k, v):
    s = (q @ k.transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    hidden = torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1)
    return torch.softmax(s.masked_fill(hidden, float("-inf")), -1) @ v


@pytest.mark.parametrize("used", [u for u in itertools.product([False, True], repeat=3) if any(u)])
def test_double_backward_with_directions_for_some_gradients(used):
    """A Hessian-vector product along some of dQ, dK, dV (the others have no gradient), with and without a term in the output
    itself: against the same chain in float64. The fp32 gate of the kernels, 1e-4."""
    import fhog
    g = torch.Generator().manual_seed(61)
    base = [torch.randn(2, 70, 64, generator=g).cuda() for _ in range(4)]
    dirs = [torch.randn(2, 70, 64, generator=g).cuda() for _ in range(3)]

    def grads(attn, cast, with_output):
        q, k, v, w = (cast(t).clone().requires_grad_(True) for t in base)
        out = attn(q, k, v)
        first = torch.autograd.grad(out, (q, k, v), w, create_graph=True)
        loss = sum((f * cast(d)).sum() for f, d, u in zip(first, dirs, used) if u)
        if with_output:
            loss = loss + out.square().sum()
        return torch.autograd.grad(loss, (q, k, v, w), allow_unused=True)

    for with_output in (False, True):
        got = grads(lambda q, k, v: fhog.attention(q, k, v, True), lambda t: t, with_output)
        want = grads(_torch_attention, lambda t: t.double(), with_output)
        for name, a, b in zip("qkvw", got, want):
            b = torch.zeros_like(base[0]) if b is None else b     # a gradient that vanishes identically
            a = torch.zeros_like(base[0]) if a is None else a
            if b.abs().max() == 0:
                assert a.abs().max() == 0, name
            else:
                assert normalised_max_error(a, b) < 1e-4, (used, with_output, name)
