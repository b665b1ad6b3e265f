"""The decode kernels' row chunks (decode.hip, ROWS) at the few-pair calls that
run them: slots of 1 to 41 rows (not multiples of the four staged at a time),
one and two row blocks a workgroup, 24 K tiles of the down projection, split
activation rows, every expert in every token, and one pair past the line.

Against the experts in float64, element-wise: a sum of K products in fp32 is
within K 2^-24 sum |w x| of the exact one; the SwiGLU activation moves by at
most 1.1 (|u| dg + |silu(g)| du) plus its rounding (2^-8 for bf16, 2^-15 for
hi + lo halves, which also cover the hardware exp2 and reciprocal); the down
projection carries that through |W_down| and adds its own sum's error.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest

from test_gpu_stream import routes

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# (H, I, rows of each expert, top_k, split activation)
CASES = {
    "t5": (1024, 512, [1, 4], 1, False),
    "k2": (512, 384, [5, 1, 4, 2], 2, False),
    "one_expert_t12": (4096, 256, [12], 1, False),
    "one_expert_t41": (7168, 128, [41], 1, False),
    "k56_tiles": (7168, 256, [13, 9, 0, 8], 1, False),
    "all_experts": (4096, 3072, [6, 6, 6, 6], 4, False),
    "split": (2048, 768, [5, 4, 9], 1, True),
    "split_24_tiles": (3584, 3072, [7, 3, 1, 1], 1, True),
    "past_the_line": (2048, 768, [5, 9, 10], 1, False),
}


@pytest.fixture(scope="module")
def hip():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import k3x_amd
    ctx = k3x_amd.Context(0)
    yield k3x_amd, ctx
    ctx.close()


@pytest.mark.parametrize("name", list(CASES))
def test_few_pair_calls(hip, name):
    k3x, ctx = hip
    H, I, counts, K, split = CASES[name]
    E, ids = len(counts), routes(counts, K)
    T = ids.shape[0]
    print(f"[gpu-test] few pairs {name}: H={H} I={I} T={T} K={K} rows {counts}", flush=True)
    sys.stdout.flush()
    bank = k3x.Bank(ctx, k3x.LayerShape(H, I, E, 0))
    bank.fill_synthetic(500 + len(name), 119, 123)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(len(name))
    x = torch.randn((T, H), device="cuda:0", generator=g).bfloat16()
    w = torch.rand((T, K), device="cuda:0", generator=g) + 0.1
    out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
    taps = dict(act=torch.empty((T * K, I), dtype=torch.bfloat16, device="cuda:0"),
                expert_out=torch.empty((T, K, H), device="cuda:0"))
    params = k3x.make_params(T, K, 1.0, flags=k3x.FLAG_SPLIT_ACT if split else 0)
    k3x.check(k3x.moe_forward_routed(ctx, bank, params, x, torch.from_numpy(ids.view(np.int32)).cuda(),
                                     w, out, taps=taps), "forward")
    k3x.check(ctx.synchronize(), "synchronize")
    row = 0
    for e in range(E):
        if not counts[e]:
            continue
        gate, up, down = (bank.dequant_rows(e, m, 0, I if m < 2 else H).double() for m in range(3))
        tok, slot = (torch.from_numpy(v).cuda() for v in np.nonzero(ids == e))
        xe = x[tok].double()
        gv, uv = xe @ gate.t(), xe @ up.t()
        eps = H * 2.0 ** -24
        dg, du = eps * (xe.abs() @ gate.abs().t()), eps * (xe.abs() @ up.abs().t())
        silu = gv / (1 + torch.exp(-gv))
        act = silu * uv
        dact = 1.1 * (uv.abs() * dg + silu.abs() * du + dg * du) + \
            (2.0 ** -15 if split else 2.0 ** -8) * act.abs() + 1e-30
        if not split:
            got = taps["act"][row:row + counts[e]].double()
            assert ((got - act).abs() <= dact).all(), (name, e, "act")
        y = act @ down.t()
        dy = dact @ down.abs().t() + I * 2.0 ** -24 * ((act.abs() + dact) @ down.abs().t())
        assert ((taps["expert_out"][tok, slot].double() - y).abs() <= dy).all(), (name, e, "out")
        row += counts[e]
    y = taps["expert_out"].double()
    mix = (w.double().unsqueeze(2) * y).sum(1)
    assert ((out.double() - mix).abs() <= 2.0 ** -8 * mix.abs() +
            2.0 ** -20 * (w.double().unsqueeze(2) * y.abs()).sum(1) + 1e-30).all()
    bank.close()
