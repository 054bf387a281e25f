"""Prompt-sized calls with and without a gradient: one result, bit for bit, and the gradient of the dense product.

The weight tile is bit-exact, so ``grad @ weight`` (the very call the node makes) is the gradient's reference where one
linear is looked at; the fused module's is float64, with three bf16 roundings in a row (2^-6).
"""

import gc

import pytest
import torch
from torch.utils.checkpoint import checkpoint

from visionrl_amd import linear as linear_mod
from visionrl_amd import ops
from visionrl_amd.linear import Int4GateUpSiLU, Int4Linear

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.fixture(scope="module", autouse=True)
def _groups_let_go():
    """Grouped modules hold each other, and their GPU tensors, in cycles."""
    yield
    gc.collect()


def _linear(gen, K, N, G=128, bias=False):
    groups = K // G
    zeros = torch.randint(0, 16 ** min(groups, 7), (N, (groups + 7) // 8), generator=gen).to(torch.int32)
    words = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), generator=gen, dtype=torch.int64).to(torch.int32)
    scales = (torch.randn(N, groups, generator=gen) * 0.02).to(torch.bfloat16)
    b = torch.randn(N, generator=gen).to(torch.bfloat16).to(DEV) if bias else None
    return Int4Linear.from_packed(words.to(DEV), scales.to(DEV), zeros.to(DEV), G, bias=b)


def _layer(seed=0, K=512, wide=768, inter=1032):
    gen = torch.Generator().manual_seed(seed)
    q, k, v = _linear(gen, K, wide, bias=True).prepack_(), _linear(gen, K, 512).prepack_(), _linear(gen, K, 512).prepack_()
    q.group_with(k, v)
    return gen, (q, k, v, _linear(gen, K, 640, 32), Int4GateUpSiLU(_linear(gen, K, inter), _linear(gen, K, inter)))


def _input(gen, *shape):
    return torch.randn(*shape, generator=gen).to(torch.bfloat16).to(DEV)


@pytest.fixture
def launches(monkeypatch):
    calls, real = [], ops.int4_gemm
    monkeypatch.setattr(linear_mod.ops, "int4_gemm", lambda *a: calls.append(len(a[1])) or real(*a))
    return calls


@pytest.mark.parametrize("rows", [33, 500, 1664, 2048, 2049, 4095, 4096])
def test_results_are_the_same_bits_with_and_without_a_gradient(rows):
    gen, modules = _layer(rows)
    x = _input(gen, rows, 512)
    with torch.no_grad():
        want = [m(x) for m in modules]
    xg = x.clone().requires_grad_()
    got = [m(xg) for m in modules]
    assert all(y.requires_grad and torch.equal(y, w) for y, w in zip(got, want))
    for m, y in zip(modules[:4], got):
        g = _input(gen, *y.shape)
        assert torch.equal(torch.autograd.grad(y, xg, g)[0], g @ m.dequantize())     # each on its own, in any order


def test_fused_module_and_its_gradient_match_float64(launches):
    gen, (*_, mlp) = _layer(1)
    w = ops.int4_dequant(mlp.qweight, mlp.scales, mlp.qzeros, 128).double()
    for shape in ((2, 300, 512), (4100, 512)):
        x = _input(gen, *shape).requires_grad_()
        ref = x.detach().double().requires_grad_()
        gate, up = (ref @ w.T).chunk(2, -1)
        want, got = torch.nn.functional.silu(gate) * up, mlp(x)
        grad = _input(gen, *got.shape)
        got.backward(grad), want.backward(grad.double())
        rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()
        assert rel(got, want) < 2.0 ** -8 and rel(x.grad, ref.grad) < 2.0 ** -6
    assert launches == [1, 1]


def test_a_group_shares_its_launch_under_a_gradient(launches):
    gen, (q, k, v, *_) = _layer(2)
    x = _input(gen, 3, 40, 512).requires_grad_()
    ys = q(x), k(x), v(x)
    assert launches == [3]
    torch.autograd.grad(ys[1].float().sum(), x)            # a sibling's graph is its own
    torch.autograd.grad(ys[0].float().sum(), x)
    q(x)                                                   # k is never called: nothing holds what led to x
    inner = torch.ones(1, device=DEV, requires_grad=True)
    led = x.detach() * inner.to(torch.bfloat16)
    q(led)
    import weakref
    gone = weakref.ref(led)
    del led
    assert gone() is None
    with torch.no_grad():                                  # made under a gradient, taken without one, and back
        q(x)
    assert k(x).requires_grad and launches[-1] == 3
    q(x)
    with torch.no_grad():
        assert not v(x).requires_grad and launches[-1] == 3


def test_gradients_of_every_kind():
    gen, (q, k, _, o, mlp) = _layer(3)
    x = _input(gen, 100, 512).requires_grad_()
    for m in (o, mlp):
        y = m(x)
        g = _input(gen, *y.shape)
        want, = torch.autograd.grad(y, x, g, retain_graph=True)
        batched, = torch.autograd.grad(y, x, torch.stack([g, 2 * g]), retain_graph=True, is_grads_batched=True)
        close = lambda a, b: torch.allclose(a.float(), b.float(), rtol=2.0 ** -5, atol=2.0 ** -5 * b.float().abs().max().item())
        assert close(batched[0], want) and close(batched[1], 2 * want)
        gg = g.clone().requires_grad_()
        first, = torch.autograd.grad(y, x, gg, create_graph=True, retain_graph=True)
        again, = torch.autograd.grad(first.float().sum(), gg, retain_graph=True)
        dense, = torch.autograd.grad(y.float() @ torch.ones(y.shape[1], 1, device=DEV), x, torch.ones(100, 1, device=DEV),
                                     retain_graph=True)
        assert again.shape == g.shape and close(first, want) and dense.shape == x.shape
        with torch.autograd.graph.save_on_cpu():
            y2 = m(x)
        assert close(torch.autograd.grad(y2, x, g)[0], want)
        with torch.autocast("cuda", torch.float16):        # a backward called under another autocast stays in bf16
            got, = torch.autograd.grad(y, x, g, retain_graph=True)
        assert torch.equal(got, want) if m is o else close(got, want)    # (SiLU's then goes through torch operators)
    second, = torch.autograd.grad(torch.autograd.grad(mlp(x).float().sum(), x, create_graph=True)[0].float().sum(), x)
    assert bool(second.float().abs().sum() > 0)


@pytest.mark.parametrize("reentrant", [True, False])
def test_checkpointed_layers_repeat_their_results(reentrant):
    gen, (q, k, v, o, mlp) = _layer(4)
    seen = []

    def block(t):
        ys = q(t), k(t), v(t), o(t), mlp(t)
        seen.append([y.detach() for y in ys])
        return sum(y.float().sum(-1) for y in ys)

    x = _input(gen, 200, 512).requires_grad_()
    plain, = torch.autograd.grad(block(x).sum(), x)
    checkpoint(block, x, use_reentrant=reentrant).sum().backward()
    assert torch.equal(x.grad, plain)
    assert len(seen) >= 2 and all(torch.equal(a, b) for other in seen[1:] for a, b in zip(seen[0], other))


def test_results_are_not_handed_across_a_capture(launches):
    """A leader's captured launch has computed nothing yet when the sibling is called outside the graph."""
    gen, (q, k, v, *_) = _layer(5)
    x = _input(gen, 64, 512)
    with torch.no_grad():
        want = q(x), k(x), v(x)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            with torch.cuda.graph(graph, stream=side):
                q(x)
            n = len(launches)
            assert torch.equal(k(x), want[1]) and len(launches) == n + 1
        torch.cuda.synchronize()


def test_a_default_device_changes_no_route(launches):
    from torch.overrides import TorchFunctionMode

    class Watching(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    gen, (q, k, v, o, mlp) = _layer(6)
    x = _input(gen, 64, 512)
    with torch.no_grad():
        want = o(x), mlp(x)
        n = len(launches)
        for device in ("cpu", "cuda:0"):
            with torch.device(device):
                assert torch.equal(o(x), want[0]) and torch.equal(mlp(x), want[1])
        assert len(launches) == n + 4
        with torch.device("cpu"), Watching():              # another mode sees the torch operators, as before
            o(x)
        assert len(launches) == n + 4
    with torch.device("cpu"):
        xg = x.clone().requires_grad_()
        y = mlp(xg)
        assert torch.equal(y, want[1])
        y.float().sum().backward()
    assert xg.grad.device == x.device


@pytest.mark.parametrize("rows", [64, 600])
def test_a_kept_dense_weight_means_library_products(rows, launches):
    """With and without a gradient, at widths where a module without the copy takes the launch."""
    gen, (q, k, v, o, mlp) = _layer(7)
    x = _input(gen, rows, 512)
    with torch.no_grad():
        o(x), mlp(x)
        assert launches == [1, 1]
        o.keep_dense_(), mlp.keep_dense_()
        dense = torch.nn.functional.linear(x, o.dequantize())
        fused = ops.silu_mul(torch.nn.functional.linear(x, ops.int4_dequant(*mlp._canonical(), 128)))
        assert torch.equal(o(x), dense) and torch.equal(mlp(x), fused)
        k.keep_dense_()                                    # one of a group: every member on its own
        q(x), v(x)
        assert torch.equal(k(x), torch.nn.functional.linear(x, k.dequantize()))
    assert launches == [1, 1, 1, 1]
    xg = x.clone().requires_grad_()
    assert torch.equal(o(xg), dense) and torch.equal(mlp(xg), fused) and launches == [1, 1, 1, 1]
