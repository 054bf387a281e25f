"""Prompt-sized int4 products (``vrl_int4_gemm_bf16``) against the same product over the dequantised weight.

The weight tile is bit-exact (``test_gpu_parity``), so the reference is a float64 product over it.  Tolerance: one
bf16 rounding of the result (2^-8 relative covers it) and the worst case of K fp32 additions, K 2^-24 sum |x w|;
the fused form carries both operands' sums through ``silu(g) * u`` (|silu'| < 1.1) and 2^-18 for exp and divide.
"""

import ctypes
import gc

import pytest
import torch

from visionrl_amd import _lib, ops
from visionrl_amd import linear as linear_mod
from visionrl_amd.linear import Int4GateUpSiLU, Int4Linear


@pytest.fixture(scope="module", autouse=True)
def _groups_let_go():
    """Grouped modules hold each other, and their GPU tensors, in cycles."""
    yield
    gc.collect()


def _triple(gen, K, N, G, dev):
    groups = K // G
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31, s, generator=gen, dtype=torch.int64).to(torch.int32)
    zeros = words(N, (groups + 7) // 8)
    if groups % 8:
        zeros[:, -1] &= (1 << (4 * (groups % 8))) - 1
    scales = (torch.randn(N, groups, generator=gen) * 0.02).to(torch.bfloat16)      # negative scales are legal
    return tuple(t.to(dev) for t in (words(N, K // 8), scales, zeros))


def _reference(x, triple, G, fused):
    w = ops.int4_dequant(*triple, G).double()
    K = x.shape[1]
    ref, eps = x.double() @ w.T, K * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    if fused:
        (g, u), (eg, eu) = ref.chunk(2, 1), eps.chunk(2, 1)
        s = torch.nn.functional.silu(g)
        ref, eps = s * u, 1.1 * eg * (u.abs() + eu) + s.abs() * eu + 2.0 ** -18 * (s * u).abs()
    return ref, eps + 2.0 ** -8 * ref.abs()


# M, N, K, G, fused, n, and the tile whose build the launch takes for them at 256 CUs ("s": waves split K)
CASES = [
    (33, 64, 256, 128, False, 1, "32x64k"),          # one row into the second tile
    (64, 2048, 2048, 128, False, 1, "32x32"),
    (65, 2050, 512, 32, False, 1, "32x32"),         # odd widths: narrow stores, a ragged last tile
    (40, 17, 256, 64, False, 3, "32x64k"),
    (70, 128, 4096, 32, False, 1, "32x32"),         # the largest tables of scales
    (500, 2048, 256, 128, False, 1, "64x64"),
    (600, 1537, 512, 64, False, 1, "64x64"),
    (300, 2048, 2048, 128, False, 3, "64x128"),
    (500, 3001, 512, 32, False, 1, "64x128"),
    (257, 2047, 256, 256, False, 3, "64x128"),
    (200, 2 * 1000, 256, 128, True, 1, "64x64"),
    (129, 2 * 77, 512, 32, True, 1, "32x64"),
    (33, 2 * 5632, 2048, 128, True, 1, "64x64"),
    (512, 3000, 512, 64, False, 2, "128x128s"),
    (300, 1000, 384, 128, False, 1, "128x128s"),    # K not a multiple of 256: the tiles with shorter chunks
    (130, 1000, 128, 128, False, 1, "128x128s"),    # one chunk
    (48, 96, 128, 32, True, 1, "128x128s"),
    (1664, 2048, 512, 128, False, 3, "128x128"),    # more tiles than CUs
    (600, 2500, 5632, 32, False, 1, "128x128"),     # the other builds' tables do not fit
    (2047, 2 * 1500, 256, 256, True, 1, "128x128"),
    (160, 2047, 1024, 128, False, 1, "32x64"),
    (150, 1000, 512, 64, False, 3, "32x64"),        # one chunk
    (129, 2 * 4001, 256, 128, True, 1, "64x128"),
    (40, 100, 11264, 32, False, 1, "32x32"),        # tables that leave room for two chunks only
    (160, 2048, 5632, 32, False, 1, "32x64"),
    (45, 2 * 100, 5632, 32, True, 1, "32x64"),
    (512, 2048, 5632, 32, False, 1, "64x64"),
    (64, 2 * 5632, 5632, 32, True, 1, "64x64"),
    (4100, 2 * 1700, 512, 64, True, 1, "256x256"),  # ragged both ways
    (4090, 3500, 256, 128, False, 1, "256x256"),
    (511, 16000, 384, 32, False, 2, "256x256"),
]


def _build(M, N, K, G, fused, n, cus=256):
    """The library's choice of tile, restated: rows and columns, chunk of K, waves, blocks of 16 x 16 per wave."""
    builds = {"32x32": (32, 32, 512, 16, 2), "32x64": (32, 64, 512, 16, 4), "32x64k": (32, 64, 256, 8, 2),
              "64x64": (64, 64, 256, 8, 8) if fused else (64, 64, 256, 16, 4), "64x128": (64, 128, 256, 16, 8),
              "128x128s": (128, 128, 128, 8, 16), "128x128": (128, 128, 64, 4, 0), "256x256": (256, 256, 64, 8, 0)}
    widths = [N + 16 * i for i in range(n)]

    def tiles(name):
        bm, bn = builds[name][:2]
        return sum(-(-M // bm) * -(-(w // 2 if fused else w) // (bn // 2 if fused else bn)) for w in widths)

    def fits(name):     # two chunks at least and the table of scales; where waves split K, their partial tiles over both
        bm, bn, kc, waves, blocks = builds[name]
        lds = 2 * (bm * kc * 2 + bn * kc // 2) + bn * (K // G) * 4
        return K % kc == 0 and max(lds, waves * blocks * 1024) <= 160 * 1024

    for name in (["32x64"] if fused else ["32x32", "32x64", "32x64k"]) + ["64x64", "64x128", "128x128s"]:
        if fits(name) and tiles(name) <= cus:
            return name
    if fits("256x256") and tiles("256x256") * 100 >= -(-tiles("256x256") // cus) * cus * 85:
        return "256x256"
    return "128x128"


def test_every_build_of_the_launch_has_a_case():
    for *shape, build in CASES:
        assert _build(*shape) == build, shape
    reached = {(build, fused) for _, _, _, _, fused, _, build in CASES}
    both = {"32x64", "64x64", "64x128", "128x128s", "128x128", "256x256"}
    assert reached == {(b, False) for b in both | {"32x32", "32x64k"}} | {(b, True) for b in both}


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,G,fused,n", [case[:6] for case in CASES])
def test_prompt_gemm_matches_dequantised_product(M, N, K, G, fused, n):
    gen = torch.Generator().manual_seed(M + N + K)
    dev = torch.device("cuda:0")
    triples = [_triple(gen, K, N + 16 * i, G, dev) for i in range(n)]
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(dev)
    ys = ops.int4_gemm(x, triples, G, fused)
    assert ys is not None
    again = ops.int4_gemm(x, triples, G, fused)
    for y, y2, t in zip(ys, again, triples):
        ref, tol = _reference(x, t, G, fused)
        assert y.shape == ref.shape and torch.equal(y, y2)
        assert bool(((y.double() - ref).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("K,N,G,tile", [(256, 300, 32, "32x64k"), (256, 2000, 32, "64x64"), (512, 800, 128, "32x64"), (512, 4000, 128, "64x128"), (384, 2000, 64, "128x128s"),
                                        (2048, 9000, 128, "128x128"), (7680, 4500, 32, "128x128")])
@pytest.mark.parametrize("largest", [116, 123])   # scales below 2^117 take the plain rebuild, a larger one the other
def test_prompt_gemm_weights_over_the_range_of_scales(K, N, G, tile, largest):
    """Rows with a single one give the weights themselves: the bits of the dequantised tile, at scales of every exponent
    (15 * 1.98 * 2^123 is still one that a bf16 holds).  K = 7680 in groups of 32: the table fills LDS, the other form."""
    gen = torch.Generator().manual_seed(K + N + largest)
    dev, M = torch.device("cuda:0"), 512
    assert _build(M, N, K, G, False, 1) == tile
    qw, _, qz = _triple(gen, K, N, G, dev)
    exponents = torch.randint(-126, 101, (N, K // G), generator=gen)
    exponents[N // 2:N // 2 + 3] = largest
    scales = torch.ldexp((1 + 0.98 * torch.rand(N, K // G, generator=gen)) * (1 - 2 * torch.randint(0, 2, (N, K // G), generator=gen)),
                         exponents).to(torch.bfloat16).to(dev)
    at = torch.randint(0, K, (M,), generator=gen)
    x = torch.zeros(M, K, dtype=torch.bfloat16)
    x[torch.arange(M), at] = 1
    (y,) = ops.int4_gemm(x.to(dev), [(qw, scales, qz)], G, False)
    assert torch.equal(y, ops.int4_dequant(qw, scales, qz, G)[:, at.to(dev)].T)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_prompt_gemm_scales_that_are_no_numbers(bad):
    """They make their own output column no number, and no other."""
    gen = torch.Generator().manual_seed(11)
    dev, K, N = torch.device("cuda:0"), 512, 700
    qw, scales, qz = _triple(gen, K, N, 128, dev)
    x = torch.randn(100, K, generator=gen).to(torch.bfloat16).to(dev)
    (clean,) = ops.int4_gemm(x, [(qw, scales, qz)], 128, False)
    scales[333, 1] = bad
    (y,) = ops.int4_gemm(x, [(qw, scales, qz)], 128, False)
    keep = torch.arange(N, device=dev) != 333
    assert bool(y[:, 333].isnan().all()) and torch.equal(y[:, keep], clean[:, keep])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,G", [
    (129, 2 * 77, 512, 32), (33, 2 * 5632, 2048, 128), (700, 2 * 2050, 512, 128), (1664, 2 * 5632, 256, 128),
    (4100, 2 * 1700, 512, 64),
])
def test_fused_launch_keeps_the_product_beside_the_result(M, N, K, G):
    gen, dev = torch.Generator().manual_seed(M), torch.device("cuda:0")
    triple = _triple(gen, K, N, G, dev)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(dev)
    products = []
    y, = ops.int4_gemm(x, [triple], G, True, products)
    assert torch.equal(y, ops.int4_gemm(x, [triple], G, True)[0])
    ref, tol = _reference(x, triple, G, False)
    assert products[0].shape == (M, N) and bool(((products[0].double() - ref).abs() <= tol).all())


@pytest.mark.gpu
def test_prompt_gemm_leaves_other_operands_to_the_general_route():
    gen, dev = torch.Generator().manual_seed(3), torch.device("cuda:0")
    x = torch.randn(64, 360, generator=gen).to(torch.bfloat16).to(dev)
    assert ops.int4_gemm(x, [_triple(gen, 360, 32, 40, dev)], 40) is None            # no MFMA form
    flat = torch.randn(64 * 256 + 1, generator=gen).to(torch.bfloat16).to(dev)
    triple = _triple(gen, 256, 32, 128, dev)
    shifted = flat[1:].view(64, 256)
    assert ops.int4_gemm(shifted, [triple], 128) is None                             # misaligned view
    module = Int4Linear.from_packed(*_triple(gen, 256, 512, 128, dev), 128)
    assert torch.equal(module(shifted), torch.nn.functional.linear(shifted, module.dequantize()))
    big = _triple(gen, 16384, 40000, 32, dev)                                        # scales beyond LDS
    x = torch.randn(400, 16384, generator=gen).to(torch.bfloat16).to(dev)
    assert ops.int4_gemm(x, [big], 32) is None


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [33, 600, 2048, 2049, 4095, 4096])
def test_modules_match_float64_on_both_sides_of_every_line(rows):
    """On the library's route gate and up are rounded to bf16 before SiLU: up to 2^-8 of each (eight significant bits,
    so half a unit in the last place is 2^-8 of a value just above a power of two), through |silu'| < 1.1 and |silu|."""
    gen, dev = torch.Generator().manual_seed(rows), torch.device("cuda:0")
    bias = torch.randn(768, generator=gen).to(torch.bfloat16).to(dev)
    triple = _triple(gen, 512, 768, 128, dev)
    linear = Int4Linear.from_packed(*triple, 128, bias=bias)
    halves = [_triple(gen, 512, 520, 64, dev) for _ in range(2)]
    mlp = Int4GateUpSiLU(*(Int4Linear.from_packed(*t, 64) for t in halves))
    x = torch.randn(1, rows, 512, generator=gen).to(torch.bfloat16).to(dev)
    with torch.no_grad():
        y, h = linear(x), mlp(x)
    assert y.shape == (1, rows, 768) and h.shape == (1, rows, 520)
    ref, tol = _reference(x[0], triple, 128, False)
    ref = ref + bias.double()                              # the bias is added in bf16: a second rounding
    assert bool(((y[0].double() - ref).abs() <= tol + 2.0 ** -8 * ref.abs() + 2.0 ** -8 * tol).all())
    both = tuple(torch.cat(ts) for ts in zip(*halves))
    ref, tol = _reference(x[0], both, 64, True)
    g, u = _reference(x[0], both, 64, False)[0].chunk(2, 1)
    tol = tol + 2.0 ** -8 * (1.1 * (g * u).abs() + torch.nn.functional.silu(g).abs() * u.abs()) * (1 + 2.0 ** -7)
    assert bool(((h[0].double() - ref).abs() <= tol).all())


@pytest.mark.gpu
def test_prompt_calls_of_a_group_share_one_launch(monkeypatch):
    gen, dev = torch.Generator().manual_seed(5), torch.device("cuda:0")
    q, k, v = (Int4Linear.from_packed(*_triple(gen, 256, n, 128, dev), 128).prepack_() for n in (768, 512, 512))
    x = torch.randn(2, 50, 256, generator=gen).to(torch.bfloat16).to(dev)
    alone = [m(x) for m in (q, k, v)]
    q.group_with(k, v)
    calls = []
    real = ops.int4_gemm
    monkeypatch.setattr(linear_mod.ops, "int4_gemm", lambda *a: calls.append(1) or real(*a))
    for want, m in zip(alone, (q, k, v)):
        assert torch.equal(m(x), want)
    assert len(calls) == 1
    q(x)
    x.mul_(2)                                   # the input changed: nothing is handed over
    assert torch.equal(k(x), real(x.view(100, 256), [k._canonical()], 128)[0].view(2, 50, 512))
    q(x)
    k.scales.mul_(2)                            # the sibling's weight changed
    assert torch.equal(k(x), real(x.view(100, 256), [k._canonical()], 128)[0].view(2, 50, 512))
    side = torch.cuda.Stream()
    q(x)
    side.wait_stream(torch.cuda.current_stream())
    n = len(calls)
    with torch.cuda.stream(side):               # a call on another stream computes its own
        v(x)
    assert len(calls) == n + 1
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_watched_prompt_calls_stay_on_the_general_route():
    """Transforms and modes see torch operators: a tangent, a batch dimension and a dispatch mode get through."""
    gen, dev = torch.Generator().manual_seed(7), torch.device("cuda:0")
    m = Int4Linear.from_packed(*_triple(gen, 256, 512, 128, dev), 128)
    x, t = (torch.randn(40, 256, generator=gen).to(torch.bfloat16).to(dev) for _ in range(2))
    with torch.no_grad():
        dense = torch.nn.functional.linear(t, m.dequantize())
        _, tangent = torch.func.jvp(m, (x,), (t,))
        assert torch.equal(tangent, dense)
        batched = torch.func.vmap(m)(torch.stack([x, t]))
        assert torch.allclose(batched[1].float(), dense.float(), rtol=2.0 ** -7, atol=1e-3)
        from torch.utils.flop_counter import FlopCounterMode
        with FlopCounterMode(display=False) as flops:
            m(x)
        assert flops.get_total_flops() == 2 * 40 * 256 * 512


@pytest.mark.gpu
def test_prompt_gemm_replays_in_a_graph():
    gen, dev = torch.Generator().manual_seed(9), torch.device("cuda:0")
    gate, up = (Int4Linear.from_packed(*_triple(gen, 256, 512, 128, dev), 128) for _ in range(2))
    mlp = Int4GateUpSiLU(gate, up)
    x = torch.randn(40, 256, generator=gen).to(torch.bfloat16).to(dev)
    with torch.no_grad():
        mlp(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = mlp(x)
        for seed in range(3):
            x.copy_(torch.randn(40, 256, generator=gen).to(torch.bfloat16))
            graph.replay()
            want = mlp(x)
            torch.cuda.synchronize()
            assert torch.equal(y, want)


@pytest.mark.gpu
def test_narrow_weights_stay_on_the_library_route(monkeypatch):
    gen, dev = torch.Generator().manual_seed(11), torch.device("cuda:0")
    narrow, wide = (Int4Linear.from_packed(*_triple(gen, 256, n, 128, dev), 128) for n in (511, 512))
    x = torch.randn(40, 256, generator=gen).to(torch.bfloat16).to(dev)
    calls, real = [], ops.int4_gemm
    monkeypatch.setattr(linear_mod.ops, "int4_gemm", lambda *a: calls.append(1) or real(*a))
    assert torch.equal(narrow(x), torch.nn.functional.linear(x, narrow.dequantize())) and not calls
    wide(x)
    assert len(calls) == 1


def test_prompt_gemm_rejects_bad_calls():
    lib = _lib.load()
    raw = ctypes.create_string_buffer(4096 + 64)
    p = (ctypes.addressof(raw) + 15) & ~15
    table = (_lib.Problem * 2)()

    def call(n=1, **fields):
        for rec in table:
            rec.x = rec.qweight = rec.scales = rec.qzeros = rec.y = p
            rec.M, rec.N, rec.K, rec.G, rec.fused_gate_up, rec.prepacked = 64, 32, 256, 128, 0, 0
            rec.product = None
        for name, value in fields.items():
            setattr(table[n - 1], name, value)
        return lib.vrl_int4_gemm_bf16(table, n, None)

    assert lib.vrl_int4_gemm_bf16(None, 1, None) == 1003
    assert call(0) == 1001 and lib.vrl_int4_gemm_bf16(table, 9, None) == 1001
    assert call(x=None) == 1003 and call(y=p + 2) == 1002
    assert call(M=0) == 1001 and call(prepacked=1) == 1001
    assert call(2, K=512) == 1001 and call(2, G=64) == 1001 and call(2, fused_gate_up=1) == 1001
    assert call(N=33, fused_gate_up=1) == 1001
    assert call(product=p) == 1001 and call(product=p + 8, fused_gate_up=1) == 1002
    assert call(K=264, G=8) == 1005 and call(K=192, G=64) == 1005 and call(K=384, G=96) == 1005


def test_prompt_gemm_refuses_inputs_it_would_misread(monkeypatch):
    """The library is handed an address: what lies there is bf16, dense and on the device, or the call ends here."""
    monkeypatch.setattr(ops._lib, "load", lambda: pytest.fail("the library was reached"))
    triple = _triple(torch.Generator().manual_seed(1), 256, 32, 128, "cpu")
    x = torch.zeros(64, 256, dtype=torch.bfloat16)
    for bad, error in ((x, ValueError), (x.half(), TypeError), (x.float(), TypeError), (x[None], ValueError),
                       (torch.zeros(64, 512, dtype=torch.bfloat16)[:, ::2], ValueError),
                       (x[:1].expand(64, 256), ValueError)):
        with pytest.raises(error):
            ops.int4_gemm(bad, [triple], 128)
