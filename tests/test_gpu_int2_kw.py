"""GPU parity of the GEMM with K split over the waves (the automatic engine of 9 rows to
several hundred) through the C ABI, at the edges of its tiles: 32-, 64- and 128-row tiles one
row short, full and one row over, column strips of 32, 64 and 128 columns ending in one
16-column block, a K shorter than one unit per wave, and its K slices (a workspace).

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

# (M, K, N): one row over the GEMV, K of two units; ragged M and N on every
# tile height; strips of 32 / 64 / 128 columns (the planner's choice follows M N)
SHAPES = [(9, 128, 16), (16, 128, 2064), (31, 256, 4112), (32, 1408, 6160), (33, 640, 1040), (63, 512, 14352),
          (65, 1152, 8208), (127, 384, 4112), (129, 768, 2064), (200, 2048, 5136), (513, 256, 1040)]
# long K over few strips: K slices with the workspace
SPLIT = [(17, 8192, 1040), (48, 14336, 4096), (130, 8192, 528)]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,K,N", SHAPES + SPLIT)
def test_kw_parity(dev, orc, M, K, N, bf16):
    """fp32 outputs against float64 sums, and the same bits from a second call."""
    import torch
    import ternocl_amd as T
    print(f"kw M={M} K={K} N={N} bf16={bf16} ws={T.int2_gemm_ws_bytes(M, N, K)}", flush=True)
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
@pytest.mark.parametrize("M,K,N", [(11, 256, 1040), (40, 8192, 528), (100, 256, 6160), (260, 256, 4112)])
def test_kw_epilogues(dev, orc, M, K, N, bf16, postop, out_f32):
    """Every epilogue on 1, 2 and 4 columns per lane, and after a K split."""
    import torch
    import ternocl_amd as T
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
