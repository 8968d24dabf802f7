"""The block transform's stages of stride 512 and up: every number of 512-element parts
that a block can have (one, two, four, eight), also as a short last block under a larger
HB, and in place."""
from __future__ import annotations

import numpy as np
import pytest

from ternocl_amd import synth
from tests.gpu_util import dev_dt, dev_raw, host_u16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("K,HB", [(4096 + 2048, 4096), (4096 + 1024, 4096), (4096 + 512, 4096), (2048 + 1024, 2048),
                                  (1024 + 8, 1024), (1024, 2048), (16, 4096)])
def test_fwht_parts_bit_exact(dev, orc, K, HB, inplace, bf16):
    import torch
    import ternocl_amd as T
    rows = 3
    print(f"fwht parts K={K} HB={HB} inplace={inplace} bf16={bf16}", flush=True)
    g = synth.rng(K + HB)
    x = synth.activations(g, (rows, K), bf16)
    s = (g.integers(0, 2, K, dtype=np.int8) * 2 - 1).astype(np.int8)
    dx = dev_dt(x, bf16)
    dy = dx if inplace else torch.zeros_like(dx)
    T.hadamard_fwht(dx, dev_raw(s), dy, rows, K, HB, True)
    torch.cuda.synchronize()
    assert np.array_equal(host_u16(dy).reshape(rows, K), orc.fwht(x, s, rows, K, HB, True, bf16))
