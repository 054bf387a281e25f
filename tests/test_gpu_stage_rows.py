"""Staging of the activations in the launches over prepacked weights: few rows go straight to LDS in pieces of 512 k.

Sizes at the edges of that: rows on both sides of the lines (2, 4) and of 16, k that ends inside a piece or in the first
one, more pieces than waves.  Reference and tolerance: a float64 product over the bit-exact dequantised weight; one bf16 rounding (2^-8 relative
covers it) and the worst case of K fp32 additions, K 2^-24 sum |x w|.
"""

import pytest
import torch

from visionrl_amd import ops


def _triple(gen, K, N, G, dev):
    groups = K // G
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31, s, generator=gen, dtype=torch.int64).to(torch.int32)
    scales = (torch.randn(N, groups, generator=gen) * 0.02).to(torch.bfloat16)
    return tuple(t.to(dev) for t in (words(N, K // 8), scales, words(N, (groups + 7) // 8)))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 7, 15, 16, 17, 32])
@pytest.mark.parametrize("K", [128, 384, 512, 2048, 2176, 4096, 5632, 11008])
@pytest.mark.parametrize("form", ["direct", "grouped"])
def test_staged_rows(M, K, form):
    gen = torch.Generator().manual_seed(100 * M + K)
    dev, N, G = torch.device("cuda:0"), 48, 128
    launch = ops.DirectGemv if form == "direct" else ops.GroupedGemv
    triple = _triple(gen, K, N, G, dev)
    weight = ops.int4_prepack(*triple, G)
    # what an earlier launch left in LDS is no number: none of it may reach a product
    wide = ops.int4_prepack(*_triple(gen, 4096, N, G, dev), G)
    launch([(torch.full((min(M, 16), 4096), float("nan"), dtype=torch.bfloat16, device=dev), wide, False)]).launch()
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(dev)
    (y,) = launch([(x, weight, False)]).launch()
    w = ops.int4_dequant(*triple, G).double()
    ref = x.double() @ w.T
    tol = K * 2.0 ** -24 * (x.double().abs() @ w.abs().T) + 2.0 ** -8 * ref.abs()
    assert bool(((y.double() - ref).abs() <= tol).all())
