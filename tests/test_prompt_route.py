"""Which prompt-sized calls go through one launch: the sizes at which both routes were timed."""

import pytest

from visionrl_amd.linear import _launch_pays

QKV, GATE_UP = dict(products=3), dict(fused=True)


@pytest.mark.parametrize("rows,K,columns,G,kind,pays", [
    # microseconds of the launch, then of dequant + library (+ SiLU)
    (512, 2048, 3 * 2048, 128, QKV, True),         # 26, 63
    (2048, 2048, 3 * 2048, 128, QKV, True),        # 63, 91
    (1280, 4096, 3 * 4096, 128, QKV, True),        # 124, 159
    (1664, 4096, 3 * 4096, 128, QKV, False),       # 206, 194
    (1024, 2048, 3 * 2048, 32, QKV, True),         # 56, 75
    (256, 4096, 3 * 4096, 32, QKV, True),          # 56, 98
    (512, 4096, 3 * 4096, 32, QKV, False),         # 144, 117
    (512, 3072, 3 * 3072, 32, QKV, False),         # 109, 89
    (256, 11008, 3 * 1024, 64, QKV, True),         # 46, 99: one round of 64 x 64 tiles
    (512, 11008, 3 * 1024, 64, QKV, False),        # 147, 124: the tables of the builds of one round do not fit
    (2048, 2048, 2048, 128, {}, True),             # 26, 30
    (1024, 5632, 2048, 128, {}, True),             # 38, 46
    (1152, 5632, 2048, 128, {}, False),            # 58, 51
    (512, 4096, 4096, 128, {}, True),              # 28, 39
    (768, 4096, 4096, 128, {}, False),             # 45, 42
    (1280, 4096, 4096, 128, {}, False),            # 81, 53
    (512, 11008, 4096, 128, {}, True),             # 67, 85
    (1280, 11008, 4096, 128, {}, False),           # 263, 128
    (256, 11008, 4096, 64, {}, True),              # 46, 60
    (512, 11008, 4096, 64, {}, False),             # 148, 85
    (512, 5632, 2048, 32, {}, True),               # 29, 30
    (1024, 5632, 2048, 32, {}, False),             # 98, 44
    (512, 2048, 16384, 128, {}, True),             # 48, 54
    (256, 4096, 16384, 128, {}, True),             # 48, 76
    (1536, 2048, 16384, 128, {}, False),           # 115, 101
    (33, 2048, 2 * 5632, 128, GATE_UP, True),      # 16, 33
    (1664, 2048, 2 * 5632, 128, GATE_UP, True),    # 94, 104
    (3072, 2048, 2 * 5632, 128, GATE_UP, False),   # 164, 148
    (8192, 2048, 2 * 5632, 128, GATE_UP, True),    # 373, 408
    (8192, 3072, 2 * 8192, 128, GATE_UP, False),   # 708, 639
    (8192, 2048, 2 * 5632, 32, GATE_UP, False),    # 424, 411
    (512, 4096, 2 * 11008, 128, GATE_UP, True),    # 127, 131
    (1280, 4096, 2 * 11008, 128, GATE_UP, False),  # 277, 222
    (256, 4096, 2 * 11008, 32, GATE_UP, False),    # 147, 97
    (1024, 3072, 2 * 8192, 32, GATE_UP, False),    # 228, 107
])
def test_the_launch_is_taken_where_it_is_the_faster_route(rows, K, columns, G, kind, pays):
    assert _launch_pays(rows, K, columns, G, **kind) is pays
