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
    up, down = (T.kw_tile_of(3, Tk * topk, N, K, E) for N, K in ((I, H), (H, I)))
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
    (32, 4096, 4096, (32, 32, 8)),       # 13.2 / 72 / 53
    # the re-pack takes 27 - 60 us where K has few slices: it or the tiles that decode themselves
    (71, 10624, 4560, (32, 32, 8, False)),    # 73.5 re-packed / 40.4
    (366, 13696, 1488, (64, 64, 8, False)),   # 107.8 / 71.6
    (64, 5376, 21504, (64, 64, 4, True)),     # 46.5 / 52.0
]


@pytest.mark.parametrize("M,K,N,tile", BITCOS)
def test_bitcos_engine(M, K, N, tile):
    import ternocl_amd as T
    got = T.kw_tile_of(2, M, N, K)
    assert (got and (got[:3] + got[4:])[:len(tile or ())]) == tile


# (M, K, N, workspace, taken): the int2 GEMM on the MFMA GEMV (M <= 16) or the
# 128-row tiles / here
INT2 = [
    (16, 512, 2256, False, True),       # the GEMV 4.4 / 4.7, but less exact sums
    (16, 4096, 4096, False, True),      # 17 / 8.2
    (212, 9728, 13760, True, False),    # four slices of 128 x 512 tiles: 81.7 / 87.7
    (774, 10752, 3600, True, False),    # 84.0 / 91.2
    (488, 10240, 5888, True, False),    # 76.4 / 84.3
    (1236, 10752, 2400, True, False),   # 79.6 / 87.3
    (164, 2816, 32528, False, False),   # 128 x 256 tiles: 48.9 / 53.2
    (293, 6272, 22528, False, True),    # 128 x 512 tiles: 136.7 / 122.8
    (1004, 10240, 2576, False, True),   # 128 x 256 tiles: 99.3 / 81.3
    (32, 14336, 4096, True, True),      # 131 / 13
    (200, 5120, 5120, True, True),      # 50 / 25
    (512, 4096, 4096, True, True),      # 43 / 24
]


@pytest.mark.parametrize("M,K,N,ws,taken", INT2)
def test_int2_engine(M, K, N, ws, taken):
    import ternocl_amd as T
    got = T.kw_tile_of(0, M, N, K, ws_bytes=T.int2_gemm_ws_bytes(M, N, K) if ws else 0)
    assert (got is not None) == taken
