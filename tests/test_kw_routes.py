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


# (M, K, N, tile or None): the M-tiled BITCOS GEMM.  A last round of a few workgroups costs a whole
# one: the tile of 64 x 64 and eight waves these calls took at 1.1 to 2.1 rounds, against the tiles
# that decode in place (no workspace) / the re-pack and the int2 ones
BITCOS = [
    (40, 256, 33968, None),              # 21.2 / 11.1 in place / 15.6 re-packed
    (45, 640, 33952, None),              # 28.2 / 17.6 / 25.4
    (10, 128, 33584, None),              # 32 x 32: 13.3 / 8.3 / 11.7
    (102, 640, 10432, None),             # 20.2 / 17.3 / 19.7
    (459, 768, 2400, None),              # 19.6 / 18.6 / 17.6
    (32, 4096, 4096, (32, 32, 8)),       # 12.1 / 70 / 52
]


@pytest.mark.parametrize("M,K,N,tile", BITCOS)
def test_bitcos_engine(M, K, N, tile):
    import ternocl_amd as T
    for bf16 in (False, True):
        got = T.kw_tile_of(2, bf16, M, N, K)
        assert (got[:3] if got else None) == tile
