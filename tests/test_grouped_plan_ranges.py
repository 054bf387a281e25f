"""How a grouped plan of prepacked records is cut into workgroup ranges, and that short plans compute right.

The ranges are read back from the plan blob (header of four words, 72-byte records, then ``{first tile, record}``
pairs): a plan is built on the host, so this runs without a GPU.
"""

import ctypes

import numpy as np
import pytest
import torch

from visionrl_amd import _lib, ops


def _ranges(shapes, M):
    lib = _lib.load()
    raw = ctypes.create_string_buffer(4096 + 64)
    p = (ctypes.addressof(raw) + 15) & ~15
    probs = (_lib.Problem * len(shapes))()
    for rec, (K, N) in zip(probs, shapes):
        rec.x = rec.qweight = rec.scales = rec.qzeros = rec.y = p
        rec.M, rec.N, rec.K, rec.G, rec.prepacked = M, N, K, 128, 1
    size = lib.vrl_int4_grouped_plan_size(len(shapes))
    plan, info = ctypes.create_string_buffer(size), _lib.PlanInfo()
    assert lib.vrl_int4_grouped_plan_build(probs, len(shapes), plan, size, ctypes.byref(info)) == 0
    blob = np.frombuffer(plan.raw, dtype=np.uint8)
    records = blob[16:16 + 72 * len(shapes)].reshape(-1, 72)
    field = lambda at: records[:, at:at + 4].copy().view(np.int32)[:, 0]
    table = blob[16 + 72 * len(shapes):][:8 * (info.grid + 1)].copy().view(np.int32).reshape(-1, 2)
    return info, field(48), field(60), table      # K and first tile of each record, {first tile, record} per range


LAYER = [(2048, 2048)] * 4 + [(2048, 5632)] * 2 + [(5632, 2048)]


@pytest.mark.parametrize("layers,M,head", [(3, 32, False), (3, 18, True), (8, 32, True), (24, 32, True), (1, 32, False),
                                           (8, 1, False), (6, 8, True), (2, 17, False), (30, 32, False)])
def test_ranges_cover_every_tile_once(layers, M, head):
    info, K, begin, table = _ranges(LAYER * layers + ([(2048, 16384)] if head else []), M)
    starts, rec = table[:, 0], table[:, 1]
    assert starts[0] == 0 and starts[-1] == info.total_tiles and (np.diff(starts) >= 0).all()
    ends = np.append(begin[1:], info.total_tiles)
    used = starts[:-1] < starts[1:]
    assert (begin[rec[:-1]][used] <= starts[:-1][used]).all() and (starts[:-1][used] < ends[rec[:-1]][used]).all()
    if M > 16:                                     # records of K = 5632 are walked in passes: whole pieces only
        inside = used & (K[rec[:-1]] == 5632)
        assert ((starts[:-1] - begin[rec[:-1]])[inside] % 8 == 0).all()
        empty = np.flatnonzero(~used)              # and no range is left empty but at the end
        assert empty.size == 0 or empty[0] >= used.sum()


@pytest.mark.gpu
@pytest.mark.parametrize("layers,M", [(1, 18), (2, 32), (3, 32)])
def test_short_plans_compute_every_output(layers, M):
    """One bf16 rounding (2^-8 relative covers it) and the worst case of K fp32 additions."""
    gen, dev = torch.Generator().manual_seed(M), torch.device("cuda:0")
    problems, refs = [], []
    for K, N in LAYER * layers + [(5632, 2000)]:
        x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(dev)
        words = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), generator=gen, dtype=torch.int64).to(torch.int32).to(dev)
        scales = (torch.randn(N, K // 128, generator=gen) * 0.02).to(torch.bfloat16).to(dev)
        zeros = torch.randint(0, 16 ** 4, (N, (K // 128 + 7) // 8), generator=gen).to(torch.int32).to(dev)
        problems.append((x, ops.int4_prepack(words, scales, zeros, 128), False))
        w = ops.int4_dequant(words, scales, zeros, 128).double()
        refs.append((x.double() @ w.T, K * 2.0 ** -24 * (x.double().abs() @ w.abs().T)))
    for y, (ref, eps) in zip(ops.GroupedGemv(problems).launch(), refs):
        assert bool(((y.double() - ref).abs() <= eps + 2.0 ** -8 * ref.abs()).all())
