"""The wide expert GEMM (grouped_gemm.hip) at every edge of its row tiles, on
bf16 rows, split activation rows and the scaled FP4 MFMA: experts of one row
to one past each multiple of 16 around the size classes (32, 64, 96 and 128
rows of a chunk) and the odd tile counts inside them (16 | 17, 48 | 49), alone
and behind a full chunk, against the experts in float64.

Bounds.  bf16 and split rows, element-wise: a sum of K products in fp32 is
within K 2^-24 sum |w x|; the SwiGLU activation moves by at most 1.1 (|u| dg +
|silu(g)| du) plus its rounding (2^-8 for bf16, 2^-15 for hi + lo halves);
down carries that through |W_down| and adds its own sum's error.  Scaled FP4,
relative error norm an expert: rows as two E4M3 terms (2^-8 of a block's
largest), sums in a window of 2^-13 of a block's largest product, the bf16
activation: 2^-6 after both projections.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest

from test_gpu_stream import routes

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

EDGES = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 95, 96, 97, 111, 112, 113,
         127, 128, 129, 144, 145, 176, 177, 1]


@pytest.mark.parametrize("mode", ["bf16", "split_act", "scaled_fp4"])
def test_wide_row_tile_edges(mode):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import k3x_amd as k3x
    ctx = k3x.Context(0)
    H, I, K, E = 512, 1024, 2, len(EDGES)
    ids = routes(EDGES, K)
    T = ids.shape[0]
    print(f"[gpu-test] wide row tiles {mode}: T={T} E={E}", flush=True)
    sys.stdout.flush()
    assert T >= 448  # the wide GEMM's range whatever the experts
    bank = k3x.Bank(ctx, k3x.LayerShape(H, I, E, 0))
    bank.fill_synthetic(77, 119, 123)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(2)
    x = torch.randn((T, H), device="cuda:0", generator=g).bfloat16()
    w = torch.rand((T, K), device="cuda:0", generator=g) + 0.1
    out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
    taps = dict(act=torch.empty((T * K, I), dtype=torch.bfloat16, device="cuda:0"),
                expert_out=torch.empty((T, K, H), device="cuda:0"))
    flags = dict(bf16=0, split_act=k3x.FLAG_SPLIT_ACT, scaled_fp4=k3x.FLAG_SCALED_FP4)[mode]
    k3x.check(k3x.moe_forward_routed(ctx, bank, k3x.make_params(T, K, flags=flags), x,
                                     torch.from_numpy(ids.view(np.int32)).cuda(), w, out,
                                     taps=taps), "forward")
    k3x.check(ctx.synchronize(), "synchronize")
    split = mode == "split_act"
    row = 0
    for e in range(E):
        gate, up, down = (bank.dequant_rows(e, m, 0, I if m < 2 else H).double() for m in range(3))
        tok, slot = (torch.from_numpy(v).cuda() for v in np.nonzero(ids == e))
        xe = x[tok].double()
        gv, uv = xe @ gate.t(), xe @ up.t()
        silu = gv / (1 + torch.exp(-gv))
        act = silu * uv
        y = act @ down.t()
        got_act = taps["act"][row:row + EDGES[e]].double()
        got = taps["expert_out"][tok, slot].double()
        row += EDGES[e]
        if mode == "scaled_fp4":
            assert float((got_act - act).norm() / act.norm()) <= 2.0 ** -6, (e, EDGES[e], "act")
            assert float((got - y).norm() / y.norm()) <= 2.0 ** -6, (e, EDGES[e], "out")
            continue
        eps = H * 2.0 ** -24
        dg, du = eps * (xe.abs() @ gate.abs().t()), eps * (xe.abs() @ up.abs().t())
        dact = 1.1 * (uv.abs() * dg + silu.abs() * du + dg * du) + \
            (2.0 ** -15 if split else 2.0 ** -8) * act.abs() + 1e-30
        if not split:
            assert ((got_act - act).abs() <= dact).all(), (e, EDGES[e], "act")
        dy = dact @ down.abs().t() + I * 2.0 ** -24 * ((act.abs() + dact) @ down.abs().t())
        assert ((got - y).abs() <= dy).all(), (e, EDGES[e], "out")
    bank.close()
    ctx.close()
