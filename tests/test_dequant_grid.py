"""The cut of a weight into dequant tiles, built for the host from the header the launch uses."""

import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "visionrl_amd", "csrc")


@pytest.fixture(scope="module")
def grid(tmp_path_factory):
    where = tmp_path_factory.mktemp("grid")
    (where / "g.cpp").write_text('#include "dequant_grid.hpp"\n'
                                 'extern "C" void grid(int N, int K, int *out) {\n'
                                 "    const DequantGrid g = dequant_grid(N, K);\n"
                                 "    const int v[] = {g.tshift, g.segments, g.rows, g.span, g.tiles, DEQUANT_TILES};\n"
                                 "    for (int i = 0; i < 6; ++i) out[i] = v[i];\n}\n")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", where / "g.so", where / "g.cpp"], check=True)
    lib = ctypes.CDLL(str(where / "g.so"))

    def call(N, K):
        out = (ctypes.c_int * 6)()
        lib.grid(N, K, out)
        return tuple(out)

    return call


@pytest.mark.parametrize("N,K,most", [(1, 8, 0), (1025, 8, 0), (17, 24, 0), (300, 256, 0), (5, 2048, 2), (4, 2056, 0),
                                      (9, 2064 * 8, 4), (1030, 2064, 0), (1030, 2064, 50)])
def test_tiles_cover_every_word_once(grid, N, K, most):
    """``most``: row tiles of one launch, to walk the launches of a larger weight (0: the library's own)."""
    tshift, segments, rows, span, tiles, limit = grid(N, K)
    most = most or limit
    seen = np.zeros((N, K // 8), dtype=int)
    t, step = np.arange(256), 256 >> tshift
    for first in range(0, tiles, most):
        for y in range(min(tiles - first, most)):
            for x in range(segments):
                r = (x << tshift) + (t & ((1 << tshift) - 1))
                for j in range(rows):
                    n = first * span + y * rows * step + (t >> tshift) + j * step
                    ok = (r < K // 8) & (n < N)
                    np.add.at(seen, (n[ok], r[ok]), 1)
    assert (seen == 1).all()


@pytest.mark.parametrize("N,K", [((1 << 25) - 1, 1 << 15), (33_000_000, 2056 * 16), (1 << 29, 2040), (2 ** 31 - 1, 504),
                                 (511, 2 ** 31 - 8), (1, 2 ** 31 - 8), (2 ** 31 - 1, 8)])
def test_the_largest_weights_stay_within_a_launch(grid, N, K):
    """Fewer than 2^32 work-items along x, what gridDim.y takes along y, row numbers of a launch within 31 bits."""
    assert N * K < 2 ** 40
    tshift, segments, rows, span, tiles, limit = grid(N, K)
    assert segments << tshift >= K // 8 and segments * 256 < 2 ** 32
    assert span == rows * (256 >> tshift) and tiles == -(-N // span) < 2 ** 31 - limit
    assert limit < 2 ** 16 and limit * span < 2 ** 31


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,G", [(1000, 2064, 24), (1030, 2064, 48), (8197, 256, 128), (64, 40000, 32), (1023, 2048, 128)])
def test_both_builds_are_bit_exact_at_ragged_sizes(N, K, G):
    from oracle import int4_oracle as oracle
    from tests._util import bf16_to_bits, to_device
    from visionrl_amd import ops

    o = oracle.make_operands(N, 1, K, N, G)
    d = to_device(o, torch.device("cuda:0"))
    got = bf16_to_bits(ops.int4_dequant(d["qweight"], d["scales"], d["qzeros"], G))
    assert (got == oracle.dequant_bf16(o["qweight"], o["scales_bits"], o["qzeros"], G)).all()
