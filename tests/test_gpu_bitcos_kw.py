"""GPU parity of the M-tiled BITCOS GEMM with K split over the waves (9 rows to a few hundred) on
every tile that it compiles, at the tiles' edges: one row short, full and one row over, strips
ending in one 16-column block, a K of one unit per wave and less, densities from empty sign
streams to a sign a row; the call with the re-pack workspace gives the same bits as the one
without, also where the two run different kernels.

fp32 outputs against float64 sums of the same factors: K exact products added in fp32 are within
K 2^-24 sum|terms|."""
from __future__ import annotations

import numpy as np
import pytest

from ternocl_amd import formats, synth
from tests.gpu_util import allclose_report, dev_dt, dev_raw, host_f32, host_u16

pytestmark = pytest.mark.gpu

# (M, K, N): (rows, columns, waves over K, whether the workspace form re-packs) of the tile it runs
# on, asserted (None: the 128-row tiles).  The re-packed words run on the int2 engine's tile of as
# many waves over K, so the two forms' bits meet across two kernels there
TILES = {
    (9, 128, 16): None, (31, 512, 2064): (32, 32, 8, False), (33, 640, 1040): (32, 32, 8, False),
    (65, 5376, 272): (32, 32, 8, False), (200, 1024, 2064): (32, 32, 8, False),
    (33, 256, 4240): (64, 32, 8, False), (64, 1408, 4112): (64, 32, 8, False), (65, 384, 2832): (64, 32, 8, False),
    (129, 1664, 3344): (64, 64, 8, False), (300, 1664, 1680): (64, 64, 8, False),
    (65, 384, 5520): (64, 64, 4, False), (129, 768, 4112): (64, 64, 4, False),
    (193, 4096, 4624): (32, 32, 8, True), (65, 896, 8208): (64, 64, 4, True),
}


def _on_tile(T, M, K, N, tile):
    got = T.kw_tile_of(2, M, N, K)
    assert (got and got[:3] + got[4:]) == tile, f"runs on {got}"


def _run(T, torch, A, buf, S, other, bias_f, M, K, N, bf16, postop, out_f32, repack):
    dB = dev_raw(buf)
    ls = T.bitcos_pick_ls(1, N, K)
    dSR = torch.zeros(max(ls - 1, 1) * N, dtype=torch.int32, device="cuda")
    T.bitcos_slice_ranks(dB, dSR, K, N, ls)
    bias = torch.from_numpy(bias_f).cuda() if out_f32 else dev_dt(formats.f32_to_dt(bias_f, bf16), bf16)
    C = torch.empty((M, N), dtype=torch.float32 if out_f32 else (torch.bfloat16 if bf16 else torch.float16), device="cuda")
    ws = torch.empty(T.bitcos_gemm_mt_ws_bytes(K, N), dtype=torch.uint8, device="cuda") if repack else None
    T.bitcos_fp16_upcvt_gemm_mt(dev_dt(A, bf16), dB, dev_dt(S, bf16), dSR, C, dev_dt(other, bf16), bias, M, N, K, ls, ws,
                                postop, out_f32)
    torch.cuda.synchronize()
    return C


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("z", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("M,K,N", TILES)
def test_bitcos_kw_parity(dev, M, K, N, z, bf16):
    import torch
    import ternocl_amd as T
    _on_tile(T, M, K, N, TILES[M, K, N])
    print(f"bitcos kw M={M} K={K} N={N} z={z} bf16={bf16}", flush=True)
    g = synth.rng(300 + M + K + N)
    A = synth.activations(g, (M, K), bf16)
    buf, codes = synth.bitcos_weights(g, K, N, z)
    S = synth.scales(g, K, N, bf16)
    other = synth.activations(g, (M, N), bf16)
    bias_f = g.standard_normal(N).astype(np.float32) * np.float32(0.1)
    got = [host_f32(_run(T, torch, A, buf, S, other, bias_f, M, K, N, bf16, 5, True, r)) for r in (False, True, False)]
    assert np.array_equal(got[0], got[1]), "with the re-pack workspace: other bits"
    assert np.array_equal(got[0], got[2]), "not the same bits twice"
    w = codes.astype(np.float64) * np.repeat(formats.dt_to_f32(S, bf16).astype(np.float64), 128, axis=0)
    a = formats.dt_to_f32(A, bf16).astype(np.float64)
    o = formats.dt_to_f32(other, bf16).astype(np.float64)
    bound = (K + 4) * 2.0 ** -24 * (np.abs(a) @ np.abs(w) + np.abs(bias_f) + np.abs(o))
    bad = int((np.abs(got[0] - (a @ w + bias_f + o)) > bound).sum())
    assert bad == 0, f"{bad} outputs outside the fp32 sum's bound"


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("postop", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("out_f32", [False, True])
@pytest.mark.parametrize("M,K,N,tile", [(20, 256, 1040, (32, 32, 8, False)), (100, 512, 4112, (64, 64, 4, False))])
def test_bitcos_kw_epilogues(dev, orc, M, K, N, tile, bf16, postop, out_f32):
    import torch
    import ternocl_amd as T
    _on_tile(T, M, K, N, tile)
    g = synth.rng(7 + postop + M)
    A = synth.activations(g, (M, K), bf16)
    buf, _ = synth.bitcos_weights(g, K, N, 0.4)
    S = synth.scales(g, K, N, bf16)
    other = synth.activations(g, (M, N), bf16)
    bias_f = g.standard_normal(N).astype(np.float32) * np.float32(0.1)
    C = _run(T, torch, A, buf, S, other, bias_f, M, K, N, bf16, postop, out_f32, True)
    bias = bias_f if out_f32 else formats.f32_to_dt(bias_f, bf16)
    want = orc.epilogue(orc.bitcos_gold(A, buf, S, M, K, N, bf16), other, bias, postop, out_f32, bf16)
    got, ref = (host_f32(C), want) if out_f32 else (formats.dt_to_f32(host_u16(C), bf16), formats.dt_to_f32(want, bf16))
    bad, dmax = allclose_report(got, ref)
    assert bad == 0, f"{bad} bad (max |d| {dmax})"
