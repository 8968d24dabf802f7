"""The tile GEMMs' cut last round: wide tiles past the last whole round of 256 run as narrower
tiles of the same rows.  The same bits as the rows computed by calls of less than a round (an
output's sum does not depend on the tile), at a last round of 128 x 128 and of 128 x 256 tiles, a
ragged last row tile and a last column tile of 16 columns, every epilogue."""
from __future__ import annotations

import numpy as np
import pytest

from tests.gpu_util import dev_dt, dev_raw, host_f32, int2_inputs

pytestmark = pytest.mark.gpu

# wide tiles: 17 x 17 = 289 (33 cut in four), 20 x 18 = 360 (104 cut in two), 2 x 160 = 320 (64 in four)
SHAPES = [(2100, 128, 8208), (2500, 128, 8720), (256, 128, 81920)]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("postop", [0, 1, 5])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_gemm_tail_same_bits(dev, M, K, N, postop, bf16):
    import torch
    import ternocl_amd as T
    print(f"gemm tail M={M} K={K} N={N} bf16={bf16} postop={postop}", flush=True)
    A, B, S, other, bias_f = int2_inputs(12 + M, M, K, N, bf16)
    dA, dB, dS, dO, dBias = dev_dt(A, bf16), dev_raw(B), dev_dt(S, bf16), dev_dt(other, bf16), torch.from_numpy(bias_f).cuda()
    eng = T.gemv_tile(T.GEMM)
    outs = []
    for step in (M, 128):
        C = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        for m in range(0, M, step):
            n = min(step, M - m)
            T.int2_fp16_upcvt_gemm(dA[m:], dB, dS, C[m:], dO[m:], dBias, n, N, K, postop, True, tile=eng)
        torch.cuda.synchronize()
        outs.append(host_f32(C))
    assert np.array_equal(outs[0], outs[1])
