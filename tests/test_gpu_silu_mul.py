"""``silu(gate) * up`` and its gradient as one launch each, against float64.

Tolerance: one bf16 rounding (2^-8 relative covers it) and 2^-17 of the terms' magnitudes for exp, divide and the
fp32 products; where exp leaves fp32 (|gate| > 88) the result is below 2^-118 and may be zero.
"""

import pytest
import torch

from visionrl_amd import _lib, ops
from visionrl_amd.linear import Int4GateUpSiLU, Int4Linear, _silu_mul, _silu_mul_ops


@pytest.mark.gpu
@pytest.mark.parametrize("M,inter", [(1, 8), (3, 520), (33, 1000), (257, 2048), (64, 5632)])
def test_silu_mul_and_gradient_match_float64(M, inter):
    gen = torch.Generator().manual_seed(M + inter)
    gu, grad = (torch.randn(M, n, generator=gen).mul_(4).to(torch.bfloat16).to("cuda:0") for n in (2 * inter, inter))
    gu[0, :4] = torch.tensor([float("inf"), 88.5, -100.0, 0.0])
    g, u = gu.double().chunk(2, 1)
    s = torch.sigmoid(g)
    y = torch.nn.functional.silu(g) * u
    got = ops.silu_mul(gu).double()
    ok = lambda a, b, size: bool((((a - b).abs() <= 2.0 ** -8 * b.abs() + 2.0 ** -17 * size + 2.0 ** -118) | (a == b)).all())
    assert ok(got, y, y.abs())
    d = grad.double()
    back = ops.silu_mul_backward(gu, grad).double()
    finite = torch.isfinite(g)              # at infinity the derivative formula is 0 * inf, as torch's is
    dg = torch.where(finite, d * u * s * (1 + g * (1 - s)), 0.0)
    size = torch.where(finite, (d * u).abs() * s * (1 + g.abs() * (1 - s)), 0.0)
    assert ok(torch.where(finite, back[:, :inter], 0.0), dg, size)
    assert ok(back[:, inter:], d * (g * s), (d * g * s).abs())


@pytest.mark.gpu
def test_gradients_of_every_kind_reach_the_product():
    """First-order gradients come from the launch; recorded, batched and hooked ones from the torch operators."""
    gen = torch.Generator().manual_seed(1)
    gu = torch.randn(6, 1024, generator=gen).to(torch.bfloat16).to("cuda:0").requires_grad_()
    grad = torch.randn(6, 512, generator=gen).to(torch.bfloat16).to("cuda:0")
    y = _silu_mul(gu)
    close = lambda a, b: torch.allclose(a.float(), b.float(), rtol=2.0 ** -5, atol=2.0 ** -5)
    want, = torch.autograd.grad(_silu_mul_ops(gu), gu, grad)
    assert type(y.grad_fn).__name__ == "_SiLUMulBackward"
    assert close(torch.autograd.grad(y, gu, grad, retain_graph=True)[0], want)
    strided = grad.t().contiguous().t()
    assert close(torch.autograd.grad(y, gu, strided, retain_graph=True)[0], want)
    batched, = torch.autograd.grad(y, gu, torch.stack([grad, 2 * grad]), retain_graph=True, is_grads_batched=True)
    assert close(batched[0], want) and close(batched[1], 2 * want)
    first, = torch.autograd.grad(y, gu, grad, create_graph=True)
    again, = torch.autograd.grad(_silu_mul_ops(gu), gu, grad, create_graph=True)
    assert close(torch.autograd.grad(first.float().sum(), gu)[0], torch.autograd.grad(again.float().sum(), gu)[0])
    with torch.autograd.graph.save_on_cpu():
        y = _silu_mul(gu)
    assert close(torch.autograd.grad(y, gu, grad)[0], want)


@pytest.mark.gpu
def test_replay_of_the_fused_module_matches_the_explicit_product():
    gen, dev = torch.Generator().manual_seed(2), torch.device("cuda:0")
    linear = lambda: Int4Linear.from_linear(torch.nn.Linear(256, 512, bias=False).to(torch.bfloat16).to(dev), 128)
    mlp = Int4GateUpSiLU(linear(), linear())
    x = torch.randn(2, 24, 256, generator=gen).to(torch.bfloat16).to(dev).requires_grad_()
    ref = x.detach().double().requires_grad_()
    w = ops.int4_dequant(mlp.qweight, mlp.scales, mlp.qzeros, 128).double()
    g, u = (ref @ w.T).chunk(2, -1)
    want = torch.nn.functional.silu(g) * u
    got = mlp(x)
    got.float().square().sum().backward()
    want.square().sum().backward()
    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()
    assert rel(got, want) < 2.0 ** -7 and rel(x.grad, ref.grad) < 2.0 ** -6     # bf16 results, three of them in a row


@pytest.mark.gpu
def test_saved_tensor_hooks_may_hand_back_views():
    """A strided view, and one that starts between 16-byte boundaries: the gradient is that of the dense tensor."""
    gen, dev = torch.Generator().manual_seed(3), torch.device("cuda:0")
    gu = torch.randn(6, 1024, generator=gen).to(torch.bfloat16).to(dev).requires_grad_()
    grad = torch.randn(6, 512, generator=gen).to(torch.bfloat16).to(dev)
    want, = torch.autograd.grad(_silu_mul(gu), gu, grad)

    def shifted(t):
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        flat[1:] = t.flatten()
        return flat[1:].view(t.shape)

    for unpack in (lambda t: t.t().contiguous().t(), shifted):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), unpack):
            y = _silu_mul(gu * 1)
        got, = torch.autograd.grad(y, gu, grad)
        assert torch.equal(got, want)


@pytest.mark.gpu
def test_an_empty_batch_passes_forward_and_backward():
    gen, dev = torch.Generator().manual_seed(4), torch.device("cuda:0")
    linear = lambda: Int4Linear.from_linear(torch.nn.Linear(256, 512, bias=False).to(torch.bfloat16).to(dev), 128)
    mlp, proj = Int4GateUpSiLU(linear(), linear()), linear()
    for shape in ((0, 256), (2, 0, 256)):
        for module in (mlp, proj):
            x = torch.randn(shape, generator=gen).to(torch.bfloat16).to(dev).requires_grad_()
            y = module(x)
            assert y.shape == (*shape[:-1], 512)
            y.float().sum().backward()
            assert x.grad.shape == x.shape


def test_silu_mul_rejects_bad_calls():
    import ctypes

    lib = _lib.load()
    raw = ctypes.create_string_buffer(4096 + 64)
    p = (ctypes.addressof(raw) + 15) & ~15
    assert lib.vrl_silu_mul_bf16(None, p, 1, 8, None) == 1003
    assert lib.vrl_silu_mul_bf16(p, p, 0, 8, None) == 1001
    assert lib.vrl_silu_mul_bf16(p, p, 1, 12, None) == 1001
    assert lib.vrl_silu_mul_bf16(p, p + 8, 1, 8, None) == 1002
    assert lib.vrl_silu_mul_backward_bf16(p, None, p, 1, 8, None) == 1003
    assert lib.vrl_silu_mul_backward_bf16(p, p, p, 1 << 20, 1 << 11, None) == 1001


def test_silu_mul_refuses_products_it_would_misread(monkeypatch):
    """An odd width would shift every row after the first; half, strided and host tensors are refused alike."""
    monkeypatch.setattr(ops._lib, "load", lambda: pytest.fail("the library was reached"))
    gu, grad = torch.zeros(4, 32, dtype=torch.bfloat16), torch.zeros(4, 16, dtype=torch.bfloat16)
    wide = torch.zeros(4, 64, dtype=torch.bfloat16)
    for bad, error in ((gu, ValueError), (gu.half(), TypeError), (wide[:, ::2], ValueError), (gu[None], ValueError),
                       (torch.zeros(4, 33, dtype=torch.bfloat16), ValueError)):
        with pytest.raises(error):
            ops.silu_mul(bad)
        with pytest.raises(error):
            ops.silu_mul_backward(bad, grad)
    for bad in (grad.half(), grad[:, :8], grad[:2]):
        with pytest.raises(ValueError):
            ops.silu_mul_backward(gu, bad)
    # the checks in their order: the odd width is what stops a device tensor of it
    with pytest.raises(ValueError, match="odd width"):
        ops.silu_mul(torch.zeros(4, 33, dtype=torch.bfloat16))
