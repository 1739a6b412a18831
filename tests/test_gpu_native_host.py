"""GPU tier: the native host side of the entry points against the Python wrappers around the same kernels."""
import warnings

import pytest
import torch

from gpu_util import require_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _dev():
    return require_gpu()


def _make(layout, n, d, dtype, g):
    """A (2, 3, n, d) or (6, n, d) tensor lying in memory as named."""
    x = torch.randn(2, 3, n, d, generator=g).to(dtype).cuda()
    if layout == "heads_last":      # (B, N, H, d) seen as (B, H, N, d)
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if layout == "padded":          # rows 16 elements longer than d
        y = torch.zeros(2, 3, n, d + 16, dtype=dtype, device="cuda")
        y[..., :d] = x
        return y[..., :d]
    return x.flatten(0, 1) if layout == "3d" else x


@pytest.mark.parametrize("layouts", [("3d", "3d"), ("4d", "4d"), ("heads_last", "heads_last"), ("padded", "padded"), ("4d", "heads_last"),
                                     ("padded", "4d")])
@pytest.mark.parametrize("case", [(torch.bfloat16, 128, True), (torch.float32, 64, False), (torch.float16, 32, "bottom_right")])
def test_native_and_python_chains_agree_bit_for_bit(layouts, case):
    """attention() through native nodes against FlashAttention.apply, and flash_bwdbwd against its own slow path (which
    return_stats takes): same kernels on the same tensors, so the same bits, and results laid out like the inputs."""
    import fhog
    dtype, d, causal = case
    g = torch.Generator().manual_seed(65)
    q, do, ddq = (_make(layouts[0], 70, d, dtype, g) for _ in range(3))
    k, v, ddk, ddv = (_make(layouts[1], 70 if causal is True else 90, d, dtype, g) for _ in range(4))

    def chain(attn):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v, do)]
        out = attn(*leaves[:3], causal)
        first = torch.autograd.grad(out, leaves[:3], leaves[3], create_graph=True)
        second = torch.autograd.grad(first, leaves, (ddq, ddk, ddv))
        return (out, *first, *second)

    for a, b in zip(chain(fhog.attention), chain(fhog.FlashAttention.apply)):
        assert a.shape == b.shape and torch.equal(a, b)
    o, L = fhog.attention_forward(q, k, v, None, causal)
    args = (q, k, v, o, do, ddq, ddk, ddv, L, d ** -0.5)
    native, python = fhog.flash_bwdbwd(*args, causal=causal), fhog.flash_bwdbwd(*args, causal=causal, return_stats=True)[:4]
    for a, b, like in zip(native, python, (q, k, v, o)):
        assert a.shape == like.shape and a.dtype == dtype and torch.equal(a, b)


@pytest.mark.parametrize("n", [1, 2, 33])
@pytest.mark.parametrize("lie", ["heads_last", "unaligned"])
def test_gradients_that_only_look_contiguous(n, lie):
    """Gradients of both orders in layouts that is_contiguous() accepts and the kernels do not: one query that comes back through
    (B, 1, H, d), and addresses off a multiple of 16 bytes. The same bits as packed ones."""
    import fhog
    g = torch.Generator().manual_seed(66)

    def laid_out(x):
        if lie == "heads_last":
            return x.transpose(1, 2).contiguous().transpose(1, 2)
        y = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:].view(x.shape)
        return y.copy_(x)

    q, k, v, do, ddq, ddk, ddv = (torch.randn(2, 3, n, 64, generator=g).bfloat16().cuda() for _ in range(7))

    def chain(f):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v, f(do))]
        first = torch.autograd.grad(fhog.attention(*leaves[:3]), leaves[:3], leaves[3], create_graph=True)
        return (*first, *torch.autograd.grad(first, leaves, (f(ddq), f(ddk), f(ddv))))

    for a, b in zip(chain(laid_out), chain(lambda t: t)):
        assert torch.equal(a, b)


def test_third_derivatives_are_refused():
    import fhog
    q, k, v, w = (torch.randn(1, 40, 64, device="cuda").requires_grad_(True) for _ in range(4))
    first = torch.autograd.grad(fhog.attention(q, k, v), (q, k, v), w, create_graph=True)
    second = torch.autograd.grad(first[0].square().sum(), q, create_graph=True)[0]
    with pytest.raises(RuntimeError, match="differentiate twice"):
        second.sum().backward()


def test_use_on_another_stream_and_thread():
    """The native call launches on the calling thread's current stream, backward included."""
    import threading
    import fhog
    q, k, v = (torch.randn(2, 300, 64, device="cuda") for _ in range(3))

    def grads():
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        return torch.autograd.grad(fhog.attention(*leaves, True).sum(), leaves)

    want, got = grads(), []

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
            got.extend(grads())
            torch.cuda.current_stream().synchronize()

    torch.cuda.synchronize()
    t = threading.Thread(target=work)
    t.start()
    t.join()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("requires_grad", [False, True])
def test_traced_module_computes_on_new_inputs(requires_grad):
    """torch.jit.trace: the traced module computes, and differentiates where its inputs ask for it, like the function itself."""
    import fhog
    g = torch.Generator().manual_seed(74)
    q, k, v = (torch.randn(2, 70, 64, generator=g).cuda().requires_grad_(requires_grad) for _ in range(3))
    traced = torch.jit.trace(lambda a, b, c: fhog.attention(a, b, c, True), (q, k, v), check_trace=False)
    new = [torch.randn(2, 70, 64, generator=g).cuda().requires_grad_(requires_grad) for _ in range(3)]
    got, want = traced(*new), fhog.attention(*new, True)
    assert torch.equal(got, want) and got.requires_grad == requires_grad
    if requires_grad:
        w = torch.randn(2, 70, 64, generator=g).cuda()
        for a, b in zip(torch.autograd.grad(got, new, w), torch.autograd.grad(want, new, w)):
            assert torch.equal(a, b)


def test_fake_tensors_propagate_shapes():
    """Under FakeTensorMode there is no memory to launch on: the torch composition stands in, with the right shapes and types, first
    derivatives included."""
    import fhog
    from fhog.attention import TorchCompositionWarning
    from torch._subclasses.fake_tensor import FakeTensorMode
    q, k, v = (torch.randn(2, n, 64, device="cuda", dtype=torch.bfloat16) for n in (70, 90, 90))
    with FakeTensorMode() as mode, pytest.warns(TorchCompositionWarning):
        leaves = [mode.from_tensor(t).requires_grad_(True) for t in (q, k, v)]
        out = fhog.attention(*leaves)
        grads = torch.autograd.grad(out.float().sum(), leaves)
    for a, b in zip((out, *grads), (q, q, k, v)):
        assert a.shape == b.shape and a.dtype == b.dtype and a.device == b.device


@pytest.mark.parametrize("layout", ["4d", "heads_last", "padded"])
def test_saved_tensors_that_come_back_elsewhere(layout):
    """Saved-tensor hooks may hand the nodes tensors that lie at addresses off a multiple of 16 bytes: the same gradients of both
    orders as without hooks."""
    import fhog
    g = torch.Generator().manual_seed(75)
    q, k, v, do, ddq, ddk, ddv = (_make(layout, 70, 64, torch.bfloat16, g) for _ in range(7))

    def off(t):
        y = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        return y.copy_(t)

    def chain():
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v, do)]
        first = torch.autograd.grad(fhog.attention(*leaves[:3]), leaves[:3], leaves[3], create_graph=True)
        return (*first, *torch.autograd.grad(first, leaves, (ddq, ddk, ddv)))

    want = chain()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, off):
        got = chain()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_attention_backward_takes_three_dimensions_only():
    import fhog
    x, L = torch.zeros(1, 2, 40, 64, device="cuda"), torch.zeros(1, 2, 40, device="cuda")
    with pytest.raises(ValueError):
        fhog.attention_backward(x, x, x, x, x, L, 0.125, False)


def test_transforms_and_forward_mode_are_refused_by_name():
    """torch.func transforms, around wrapped or plain tensors, and dual tensors: refused with the reason, not computed and not failing
    on an address."""
    import fhog
    q, k, v = (torch.randn(2, 40, 64, device="cuda") for _ in range(3))
    for f in (lambda: torch.func.grad(lambda a: fhog.attention(a, k, v).sum())(q),
              lambda: torch.func.vmap(lambda a: fhog.attention(a, k, v))(q[None]),
              lambda: torch.func.grad(lambda a: (fhog.attention(q, k, v) * a).sum())(q)):
        with pytest.raises(RuntimeError, match="setup_context"):
            f()
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level(), pytest.raises(RuntimeError, match="(?i)forward AD|jvp"):
        fhog.attention(fwAD.make_dual(q, torch.ones_like(q)), k, v)


def test_tensors_elsewhere_or_of_other_shapes_are_refused():
    """Host memory beside device tensors, and tensors shorter than the others: errors of the wrappers (or of the torch composition that
    the first-order ones hand such calls to), before any launch."""
    import fhog
    x, short, L = torch.zeros(2, 40, 64, device="cuda"), torch.zeros(2, 33, 64, device="cuda"), torch.zeros(2, 40, device="cuda")
    host = x.cpu()
    for f in (lambda: fhog.attention(x, host, x), lambda: fhog.attention(x, x, short), lambda: fhog.attention_forward(x, x, host),
              lambda: fhog.attention_forward(x, x, short), lambda: fhog.attention_forward(x, x[:1], x[:1], use_hip=True),
              lambda: fhog.attention_backward(x, x, x, host, x, L, 0.125, False), lambda: fhog.attention_backward(x, x, x, x, short, L, 0.125, False),
              lambda: fhog.attention_backward(x, x, x, x, x, L.cpu(), 0.125, False),
              lambda: fhog.flash_bwdbwd(x, x, x, x, x, x, x, x, L.cpu(), 0.125),
              lambda: fhog.BwdBwdPlan(x, x, x, x, x, x, x, x, L.cpu(), 0.125), lambda: fhog.BwdBwdPlan(x, x, x, x, short, x, x, x, L, 0.125),
              lambda: fhog.BwdBwdPlan(x, x, short, x, x, x, x, x, L, 0.125)):
        with pytest.raises((ValueError, RuntimeError)), warnings.catch_warnings():
            warnings.simplefilter("ignore")
            f()
    with pytest.raises(TypeError):
        fhog.BwdBwdPlan(x, x, x, x, x, x.half(), x, x, L, 0.125)
