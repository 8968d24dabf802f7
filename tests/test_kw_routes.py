"""Which engine the automatic calls take, without a GPU: sizes at which a rule once chose the
slower one, with both times (graph-timed, us) beside each."""
from __future__ import annotations

import pytest

# (T, E, topk, H, I, taken): the MoE layer on 128-row tiles / on the K-over-waves tiles
MOE = [
    (256, 64, 8, 2048, 1408, False),   # 115 / 111: level
    (384, 64, 8, 2048, 1408, False),   # 123 / 145
    (512, 64, 8, 2048, 1408, False),   # 171 / 171
    (64, 256, 8, 2048, 512, False),    # 98 / 127
    (64, 128, 8, 2048, 768, False),    # 85 / 92
    (720, 128, 2, 896, 1024, False),   # 56 / 70
    (1, 128, 8, 2048, 768, True),      # 77 / 30
    (16, 128, 8, 2048, 768, True),     # 80 / 67
    (64, 64, 8, 2048, 1408, True),     # 93 / 81
    (128, 64, 8, 2048, 1408, True),    # 97 / 84
    (128, 16, 4, 3072, 1536, True),    # 122 / 61
    (256, 8, 2, 4096, 1536, True),     # 156 / 58
]


@pytest.mark.parametrize("Tk,E,topk,H,I,taken", MOE)
def test_moe_engine(Tk, E, topk, H, I, taken):
    """The layer's products (N, K) = (I, H) and (H, I) take the same engine, whichever is faster."""
    import ternocl_amd as T
    up, down = (T.kw_tile_of(3, True, Tk * topk, N, K, E) for N, K in ((I, H), (H, I)))
    assert (up is not None) == taken and (down is not None) == taken
