"""GPU parity of the GEMM with K split over the waves (the automatic engine of 9 rows to
several hundred) through the C ABI, on every tile that it compiles, at the tiles' edges, with and
without K slices (a workspace).

Gold: the oracle's restatement of compute_gold + epilogue_ref (int2_fp16_upcvt/main.cpp:79-98,
common/epilogue.hpp:98-115); fp32 outputs are compared with float64 sums: K products of exact
16-bit factors added in fp32 are within K 2^-24 sum|terms|.
"""
from __future__ import annotations

import numpy as np
import pytest

from ternocl_amd import formats
from tests.gpu_util import allclose_report, dev_dt, dev_raw, host_f32, host_u16
from tests.gpu_util import int2_gold, int2_inputs, int2_run

pytestmark = pytest.mark.gpu

# (M, K, N): (rows, columns, waves over K, K slices) of the tile it runs on, asserted, so that a
# change of the planner cannot empty the list.  Row tiles one row short, full and one row over,
# strips that end in one 16-column block, K of a unit a wave and less
TILES = {
    (9, 128, 16): (32, 32, 8, 1), (16, 128, 2064): (32, 32, 8, 1), (31, 256, 4112): (32, 32, 8, 1),
    (32, 1408, 6160): (32, 32, 8, 1), (33, 640, 1040): (32, 32, 8, 1),
    (31, 384, 8208): (32, 64, 8, 1), (33, 896, 4112): (32, 64, 8, 1), (97, 896, 2064): (32, 64, 8, 1),
    (65, 1152, 8208): (32, 128, 4, 1), (129, 384, 5520): (32, 128, 4, 1),
    (63, 512, 14352): (64, 64, 4, 1), (127, 384, 4112): (64, 64, 4, 1), (129, 768, 2064): (64, 64, 4, 1),
    (513, 256, 1040): (64, 64, 4, 1),
    (65, 896, 11536): (64, 128, 4, 1), (200, 2048, 5136): (64, 128, 4, 1),
    (300, 3072, 9744): (128, 128, 4, 1),
    # long K over few strips: K slices with the workspace
    (17, 8192, 1040): (32, 32, 8, 7), (130, 8192, 528): (32, 32, 8, 3), (129, 9216, 400): (32, 64, 8, 7),
    (48, 14336, 4096): (32, 128, 4, 4), (65, 3072, 2832): (32, 128, 4, 3), (96, 5120, 1024): (64, 64, 4, 8),
    (129, 6144, 3344): (64, 128, 4, 3), (97, 4608, 8208): (128, 128, 4, 3),
}


def _on_tile(T, M, K, N, tile):
    got = T.kw_tile_of(0, M, N, K, ws_bytes=T.int2_gemm_ws_bytes(M, N, K))
    assert (got and got[:4]) == tile, f"runs on {got}"


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,K,N", TILES)
def test_kw_parity(dev, orc, M, K, N, bf16):
    """fp32 outputs against float64 sums, and the same bits from a second call."""
    import torch
    import ternocl_amd as T
    print(f"kw M={M} K={K} N={N} bf16={bf16} ws={T.int2_gemm_ws_bytes(M, N, K)}", flush=True)
    _on_tile(T, M, K, N, TILES[M, K, N])
    A, B, S, other, bias_f = int2_inputs(81 + M + K + N, M, K, N, bf16)
    dC, dW = int2_run(T, torch, A, B, S, other, bias_f, M, K, N, bf16, 5, True)
    got = host_f32(dC).astype(np.float64)
    dC2, _ = int2_run(T, torch, A, B, S, other, bias_f, M, K, N, bf16, 5, True)
    assert np.array_equal(host_f32(dC), host_f32(dC2)), "not the same bits twice"
    if dW is not None:
        assert not dW[:T.WS_HEADER_BYTES].any().item(), "a counter was left set"
    codes = (B[:, None, :] >> (2 * np.arange(16, dtype=np.uint32))[None, :, None]) & 3
    v = np.where(codes == 3, -1.0, codes).reshape(K, N)
    w = v * np.repeat(formats.dt_to_f32(S, bf16).astype(np.float64), 128, axis=0)
    a = formats.dt_to_f32(A, bf16).astype(np.float64)
    o = formats.dt_to_f32(other, bf16).astype(np.float64)
    want = a @ w + bias_f.astype(np.float64) + o
    bound = (K + 4) * 2.0 ** -24 * (np.abs(a) @ np.abs(w) + np.abs(bias_f) + np.abs(o))
    bad = int((np.abs(got - want) > bound).sum())
    assert bad == 0, f"{bad} outputs outside the fp32 sum's bound"


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("postop", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("out_f32", [False, True])
@pytest.mark.parametrize("M,K,N,tile", [(11, 256, 1040, (32, 32, 8, 1)), (40, 8192, 528, (32, 32, 8, 7)),
                                        (100, 256, 6160, (64, 64, 4, 1)), (129, 384, 5520, (32, 128, 4, 1)),
                                        (129, 3072, 1808, (32, 128, 4, 3)), (260, 256, 4112, None)])
def test_kw_epilogues(dev, orc, M, K, N, tile, bf16, postop, out_f32):
    """Every epilogue on 1, 2 and 4 columns per lane, after a K split, and (None) on the 128-row tiles."""
    import torch
    import ternocl_amd as T
    _on_tile(T, M, K, N, tile)
    print(f"kw epilogue M={M} K={K} N={N} bf16={bf16} postop={postop} f32={out_f32}", flush=True)
    A, B, S, other, bias_f = int2_inputs(170 + postop + M, M, K, N, bf16)
    dC, _ = int2_run(T, torch, A, B, S, other, bias_f, M, K, N, bf16, postop, out_f32)
    want, _ = int2_gold(orc, A, B, S, other, bias_f, M, K, N, bf16, postop, out_f32)
    if out_f32:
        got, ref = host_f32(dC), want
    else:
        got, ref = formats.dt_to_f32(host_u16(dC), bf16), formats.dt_to_f32(want, bf16)
    bad, dmax = allclose_report(got, ref)
    assert bad == 0, f"{bad} bad (max |d| {dmax})"


@pytest.mark.parametrize("M,N,K", [(24, 4096, 4096), (48, 4096, 14336)])
def test_kw_scratch_and_alignment(dev, M, N, K):
    """A short workspace runs unsplit, an operand off its 16-byte alignment takes the engines that
    read it: results within the DT rounding of each other."""
    import torch
    import ternocl_amd as T
    A, B, S, other, bias_f = int2_inputs(5, M, K, N, True)
    dA, dB, dS = dev_dt(A, True), dev_raw(B), dev_dt(S, True)
    need = T.int2_gemm_ws_bytes(M, N, K)
    outs = []
    for ws_bytes, shift in ((need, 0), (max(0, need - 256), 0), (0, 0), (0, 2)):
        ws = torch.zeros(ws_bytes, dtype=torch.uint8, device="cuda") if ws_bytes else None
        a = torch.empty(M * K + shift, dtype=dA.dtype, device="cuda")[shift:]
        a.copy_(dA.reshape(-1))
        C = torch.empty((M, N), dtype=torch.float32, device="cuda")
        T.int2_fp16_upcvt_gemm(a, dB, dS, C, None, None, M, N, K, 0, True, ws=ws)
        torch.cuda.synchronize()
        outs.append(C)
    for C in outs[1:]:
        assert torch.allclose(outs[0], C, rtol=1e-4, atol=1e-4)
