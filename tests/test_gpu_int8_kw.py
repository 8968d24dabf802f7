"""GPU parity of the s8 x s2 GEMM with K split over the waves (5 rows to several hundred) on every
tile that it compiles, at the tiles' edges: one row short, full and one row over, strips ending
in one 16-column block, fewer groups than waves, with and without K slices (a workspace); both
quantization modes (the same bits), all four codes.

Gold: the int8 rows and scales of quant_a (bit-exact with the oracle, tests/test_gpu_int8.py) in
float64.  The group dots are exact in int32; each of a column's G = K / 128 groups adds
float(dot) (SB (1 / SA)) with four fp32 roundings, so an output is within (G + 4) 2^-24 of its
sum of |terms| (int2_via_int2_x_int8_dpas/main.cpp:113-116 is the fold)."""
from __future__ import annotations

import numpy as np
import pytest

from ternocl_amd import formats, synth
from tests.gpu_util import allclose_report, dev_dt, dev_raw, host_f32, host_u16

pytestmark = pytest.mark.gpu

# (M, K, N): (rows, columns, waves over K, K slices) of the tile it runs on, asserted (None: the
# tile engines)
TILES = {
    (5, 128, 16): None,  # (one group: the tile engine)
    (7, 256, 1040): (32, 32, 8, 1), (31, 256, 2064): (32, 32, 8, 1), (32, 1408, 4112): (32, 32, 8, 1),
    (33, 640, 1040): (32, 32, 8, 1),
    (31, 384, 8208): (32, 64, 8, 1), (65, 1152, 4112): (32, 64, 8, 1), (129, 768, 2064): (32, 64, 8, 1),
    (65, 640, 8208): (32, 64, 4, 1), (200, 2048, 5136): (32, 64, 4, 1),
    (63, 512, 8208): (64, 64, 4, 1), (65, 512, 5520): (64, 64, 4, 1),
    # K slices with the workspace
    (6, 14336, 1040): (32, 32, 8, 7), (130, 8192, 528): (32, 32, 8, 3), (300, 8192, 272): (32, 64, 8, 5),
    (65, 6144, 3088): (32, 64, 4, 3), (48, 14336, 4096): (64, 64, 4, 4),
}


def _on_tile(T, M, K, N, tile):
    got = T.kw_tile_of(1, M, N, K, ws_bytes=T.int2_int8_gemm_ws_bytes(M, N, K))
    assert (got and got[:4]) == tile, f"runs on {got}"


def _case(T, torch, seed, M, K, N, bf16):
    g = synth.rng(seed)
    A = synth.activations(g, (M, K), bf16)
    B = g.integers(0, 2**32, size=(K // 16, N), dtype=np.uint32)  # all four codes
    SB = synth.scales(g, K, N, bf16)
    dA = dev_dt(A, bf16)
    dSA = torch.zeros((K // 128, T.ldsa(M)), dtype=dA.dtype, device="cuda")
    dAq = torch.zeros((M, K), dtype=torch.int8, device="cuda")
    T.quant_a(dA, dSA, dAq, M, K)
    return B, SB, dA, dSA, dAq, dev_raw(B), dev_dt(SB, bf16)


def _ws(T, torch, M, N, K):
    need = T.int2_int8_gemm_ws_bytes(M, N, K)
    return torch.zeros(need, dtype=torch.uint8, device="cuda") if need else None


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,K,N", TILES)
def test_int8_kw_parity(dev, M, K, N, bf16):
    import torch
    import ternocl_amd as T
    _on_tile(T, M, K, N, TILES[M, K, N])
    print(f"int8 kw M={M} K={K} N={N} bf16={bf16} ws={T.int2_int8_gemm_ws_bytes(M, N, K)}", flush=True)
    B, SB, dA, dSA, dAq, dB, dSB = _case(T, torch, 900 + M + K + N, M, K, N, bf16)
    outs = []
    for mode in (0, 1, 0):
        ws = _ws(T, torch, M, N, K)
        C = torch.empty((M, N), dtype=torch.float32, device="cuda")
        T.int2_int8_gemm(dA if mode else None, None if mode else dAq, dSA, dB, dSB, C, None, None, M, N, K, 0, True, ws=ws)
        torch.cuda.synchronize()
        if ws is not None:
            assert not ws[:T.WS_HEADER_BYTES].any().item(), "a counter was left set"
        outs.append(host_f32(C))
    assert np.array_equal(outs[0], outs[1]), "the quantization modes differ"
    assert np.array_equal(outs[0], outs[2]), "not the same bits twice"
    codes = (B[:, None, :] >> (2 * np.arange(16, dtype=np.uint32))[None, :, None]) & 3
    v = np.where(codes >= 2, codes.astype(np.float64) - 4, codes.astype(np.float64)).reshape(K, N)
    sa = formats.dt_to_f32(host_u16(dSA)[:, :M], bf16).astype(np.float64)  # [G, M]
    sb = formats.dt_to_f32(SB, bf16).astype(np.float64)
    G = K // 128
    dots = np.einsum("mgk,gkn->gmn", dAq.cpu().numpy().astype(np.float64).reshape(M, G, 128), v.reshape(G, 128, N))
    terms = dots * sb[:, None, :] / sa[:, :, None]
    bad = int((np.abs(outs[0] - terms.sum(0)) > (G + 4) * 2.0 ** -24 * np.abs(terms).sum(0)).sum())
    assert bad == 0, f"{bad} outputs outside the fold's bound"


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("postop", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("out_f32", [False, True])
@pytest.mark.parametrize("M,K,N,tile", [(7, 256, 1040, (32, 32, 8, 1)), (40, 8192, 528, (32, 32, 8, 7)),
                                        (100, 384, 2064, (32, 64, 8, 1)), (65, 512, 5520, (64, 64, 4, 1)),
                                        (100, 256, 2064, None)])
def test_int8_kw_epilogues(dev, orc, M, K, N, tile, bf16, postop, out_f32):
    """Every epilogue on one and two columns per lane and after a K split, against the oracle's
    epilogue of the postop-0 fp32 sums (the same sums: the same plan)."""
    import torch
    import ternocl_amd as T
    _on_tile(T, M, K, N, tile)
    _, _, _, dSA, dAq, dB, dSB = _case(T, torch, 40 + M, M, K, N, bf16)
    g = synth.rng(postop)
    other = synth.activations(g, (M, N), bf16)
    bias_f = g.standard_normal(N).astype(np.float32) * np.float32(0.1)
    bias = bias_f if out_f32 else formats.f32_to_dt(bias_f, bf16)
    ws = _ws(T, torch, M, N, K)
    acc = torch.empty((M, N), dtype=torch.float32, device="cuda")
    T.int2_int8_gemm(None, dAq, dSA, dB, dSB, acc, None, None, M, N, K, 0, True, ws=ws)
    C = torch.empty((M, N), dtype=torch.float32 if out_f32 else dSB.dtype, device="cuda")
    dBias = torch.from_numpy(bias_f).cuda() if out_f32 else dev_dt(bias, bf16)
    T.int2_int8_gemm(None, dAq, dSA, dB, dSB, C, dev_dt(other, bf16), dBias, M, N, K, postop, out_f32, ws=ws)
    torch.cuda.synchronize()
    want = orc.epilogue(host_f32(acc), other, bias, postop, out_f32, bf16)
    got = host_f32(C) if out_f32 else formats.dt_to_f32(host_u16(C), bf16)
    bad, dmax = allclose_report(got, want if out_f32 else formats.dt_to_f32(want, bf16))
    assert bad == 0, f"{bad} bad (max |d| {dmax})"
