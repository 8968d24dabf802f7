"""GPU parity of the MoE prefill's grouped GEMMs for experts of few rows: empty experts, experts
of 1, 31, 32, 33, 64 and 70 rows, more than 64 experts (two steps of the tile search), dropped
assignments; the layer equals its stages bit for bit, and every output is within the rule of the
oracle's stage composition (tests/test_gpu_moe.py)."""
from __future__ import annotations

import numpy as np
import pytest

from ternocl_amd import formats, synth
from tests.gpu_util import allclose_report, dev_dt, dev_raw, host_u16
from tests.test_gpu_moe import _ints, _layer, _oracle_layer, _route, _weights

pytestmark = pytest.mark.gpu

# rows per expert (top-1): one 32-row tile, several, 70 experts
COUNTS = [[0, 1, 31, 32, 33, 2, 0, 5, 64, 1, 1, 1], [40, 64, 65, 33, 0, 1, 63, 30],
          [1] * 30 + [0] * 10 + [3] * 29 + [70]]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("counts", COUNTS)
def test_moe_kw_layer(dev, orc, counts, bf16):
    import torch
    import ternocl_amd as T
    E, topk, H, I = len(counts), 1, 256, 384
    g = synth.rng(50 + E)
    ids = np.repeat(np.arange(E, dtype=np.int32), counts)
    g.shuffle(ids)
    Tk = ids.size
    print(f"moe kw T={Tk} E={E} bf16={bf16}", flush=True)
    assert T.kw_tile_of(3, Tk, I, H, E) and T.kw_tile_of(3, Tk, H, I, E), "another engine runs the layer"
    X = synth.activations(g, (Tk, H), bf16)
    RW = formats.f32_to_dt(np.ones(Tk, np.float32), bf16)
    W = _weights(g, E, H, I, bf16)
    out = _layer(T, torch, X, ids, RW, Tk, E, topk, H, I, W, bf16)
    got = formats.dt_to_f32(out, bf16)
    want = formats.dt_to_f32(_oracle_layer(orc, X, ids, RW, Tk, E, topk, H, I, W, bf16, T.moe_tile_rows()), bf16)
    bad, dmax = allclose_report(got, want)
    assert bad == 0, f"{bad} of {got.size} outputs outside the rule (max |d| {dmax})"
    # the stages as separate calls: the same bits
    (Bg, Sg), (Bu, Su), (Bd, Sd) = W
    dt = torch.bfloat16 if bf16 else torch.float16
    meta, perm, inv = _route(T, ids, Tk, E)
    dX = dev_dt(X, bf16)
    U = torch.zeros((Tk, I), dtype=dt, device="cuda")
    Hs = torch.zeros((Tk, I), dtype=dt, device="cuda")
    Y = torch.zeros((Tk, H), dtype=torch.float32, device="cuda")
    O = torch.zeros((Tk, H), dtype=dt, device="cuda")
    T.int2_moe_gemm(meta, dX, perm, topk, dev_raw(Bu), dev_dt(Su, bf16), U, None, E, Tk, I, H, 0, False)
    T.int2_moe_gemm(meta, dX, perm, topk, dev_raw(Bg), dev_dt(Sg, bf16), Hs, U, E, Tk, I, H, 1, False)
    T.int2_moe_gemm(meta, Hs, None, 1, dev_raw(Bd), dev_dt(Sd, bf16), Y, None, E, Tk, H, I, 0, True)
    T.int2_moe_combine(Y, inv, dev_dt(RW, bf16), O, Tk, topk, H)
    torch.cuda.synchronize()
    assert np.array_equal(out, host_u16(O)), "the layer and its stages differ"


def test_moe_kw_dropped_ids(dev, orc):
    """Assignments outside [0, E) take no row of any tile: the layer of the others alone."""
    import torch
    import ternocl_amd as T
    Tk, E, topk, H, I, bf16 = 20, 16, 2, 256, 256, True
    g = synth.rng(9)
    X = synth.activations(g, (Tk, H), bf16)
    ids, RW = synth.moe_routing(g, Tk, E, topk, bf16)
    W = _weights(g, E, H, I, bf16)
    bad = ids.copy()
    bad[::5] = np.where(np.arange(bad[::5].size) % 2 == 0, -1, E)
    rw0 = RW.copy()
    rw0[::5] = 0
    assert T.kw_tile_of(3, Tk * topk, I, H, E) and T.kw_tile_of(3, Tk * topk, H, I, E)
    a = _layer(T, torch, X, bad, RW, Tk, E, topk, H, I, W, bf16)
    b = _layer(T, torch, X, ids, rw0, Tk, E, topk, H, I, W, bf16)
    assert np.array_equal(formats.dt_to_f32(a, bf16), formats.dt_to_f32(b, bf16))
