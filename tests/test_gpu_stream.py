"""The streaming expert GEMM (stream_gemm.hip) at the edges of its tiles,
against the experts in float64.

Routes are given (k3x_hip_moe_forward_routed) so that each expert gets a
chosen number of rows: around one row tile of 16, the 32, 48 and 64 rows of
a chunk, and past it; K extents of one to a few tiles (not multiples of the
ring), output row blocks that do not fill a workgroup, one slot a token and
two, both record layouts (a slot an expert up to four tokens, row chunks beyond),
experts of more rows than a pass, and split input and activation rows.

Bounds, element-wise: a projection's fp32 sum is within 2^-16 sum |w x| of
the float64 one (5 K tiles at most: 640 terms of 2^-24 each, doubled); the
SwiGLU activation moves by at most 1.1 (|u| dg + |silu(g)| du) plus its
rounding (2^-8 for bf16, 2^-15 for hi + lo halves, which also cover the
hardware exp2 and reciprocal); the down projection carries that through
|W_down| and adds its own sum's error.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def hip():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import k3x_amd
    ctx = k3x_amd.Context(0)
    yield k3x_amd, ctx
    ctx.close()


def routes(counts, top_k):
    """[T][top_k] ids, expert e used by counts[e] pairs, distinct within a token: the pairs
    sorted by expert and dealt to the tokens column by column."""
    pairs = np.repeat(np.arange(len(counts)), counts)
    assert len(pairs) % top_k == 0 and max(counts) <= len(pairs) // top_k
    return np.ascontiguousarray(pairs.reshape(top_k, -1).T.astype(np.uint32))


# (H, I, counts, top_k, split input, split activation)
EDGE = [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65]          # 434 pairs: row chunks
CASES = {
    "chunks": (640, 384, EDGE, 1, False, False),
    "chunks_k2": (640, 384, EDGE, 2, False, False),
    "chunks_split_act": (640, 384, EDGE, 1, False, True),
    "chunks_split_both": (384, 640, EDGE, 1, True, True),
    "chunks_split_in": (384, 640, EDGE, 1, True, False),
    "one_chunked_expert": (512, 256, [0, 300, 0], 1, False, False),
    # T <= 4: the small-route grouping's slot records.
    "slots_t4": (640, 384, [4, 3, 1], 2, False, False),
    "slots_t3_split_act": (640, 384, [3, 2, 1], 2, False, True),
    "slots_t4_split_both": (640, 384, [4, 0, 3, 1], 2, True, True),
    # 65 to 96 tokens: two row tiles, busier experts in several passes.
    "passes_t70": (640, 384, [33, 48, 64, 65], 3, False, False),
    "passes_t70_split_act": (640, 384, [33, 48, 64, 65], 3, False, True),
    "small_long": (256, 512, [1, 2, 100, 130], 1, False, False),
    "small_long_split": (256, 512, [1, 2, 100, 130], 1, True, True),
    "t16": (896, 128, [3, 4, 0, 9], 1, False, False),
    "t16_split": (896, 128, [3, 4, 0, 9], 1, True, True),
    "t25": (896, 1152, [20, 5], 1, False, True),
    "one_tile": (128, 128, [1, 3], 1, False, False),
    "k2_t17": (384, 384, [17, 1, 2, 14], 2, False, False),
}


@pytest.mark.parametrize("name", list(CASES))
def test_stream_gemm_edges(hip, name):
    k3x, ctx = hip
    H, I, counts, K, split_in, split_act = CASES[name]
    E = len(counts)
    ids = routes(counts, K)
    T = ids.shape[0]
    print(f"[gpu-test] stream gemm {name}: H={H} I={I} T={T} K={K} rows {counts}", flush=True)
    sys.stdout.flush()
    bank = k3x.Bank(ctx, k3x.LayerShape(H, I, E, 0))
    bank.fill_synthetic(1000 + len(name), 119, 123)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(len(name))
    x = torch.randn((T, H), device="cuda:0", generator=g)
    hi = x.bfloat16()
    xin, xv = hi, hi.double()
    if split_in:
        lo = (x - hi.float()).bfloat16()
        xin = torch.cat([hi, lo], 1).contiguous()
        xv = hi.double() + lo.double()
    dids = torch.from_numpy(ids.view(np.int32)).cuda()
    w = torch.rand((T, K), device="cuda:0", generator=g) + 0.1
    out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
    taps = dict(act=torch.empty((T * K, I), dtype=torch.bfloat16, device="cuda:0"),
                expert_out=torch.empty((T, K, H), device="cuda:0"),
                offsets=torch.empty(E + 1, dtype=torch.int32, device="cuda:0"),
                pair_token=torch.empty(T * K, dtype=torch.int32, device="cuda:0"),
                pair_slot=torch.empty(T * K, dtype=torch.int32, device="cuda:0"))
    flags = (k3x.FLAG_SPLIT_INPUT if split_in else 0) | (k3x.FLAG_SPLIT_ACT if split_act else 0) | \
        k3x.FLAG_GENERAL_PATH
    params = k3x.make_params(T, K, 1.0, flags=flags)
    k3x.check(k3x.moe_forward_routed(ctx, bank, params, xin, dids, w, out, taps=taps), "forward")
    k3x.check(ctx.synchronize(), "synchronize")
    off, tok, slot = (taps[n].cpu().numpy() for n in ("offsets", "pair_token", "pair_slot"))
    eps = 2.0 ** -16
    for e in range(E):
        r0, r1 = off[e], off[e + 1]
        assert r1 - r0 == counts[e]
        if not counts[e]:
            continue
        gate, up, down = (bank.dequant_rows(e, m, 0, I if m < 2 else H).double() for m in range(3))
        rows = torch.from_numpy(tok[r0:r1].astype(np.int64)).cuda()
        xe = xv[rows]
        gv, uv = xe @ gate.t(), xe @ up.t()
        dg, du = eps * (xe.abs() @ gate.abs().t()), eps * (xe.abs() @ up.abs().t())
        silu = gv / (1 + torch.exp(-gv))
        act = silu * uv
        dact = 1.1 * (uv.abs() * dg + silu.abs() * du + dg * du) + \
            (2.0 ** -15 if split_act else 2.0 ** -8) * act.abs() + 1e-30
        if not split_act:
            got = taps["act"][r0:r1].double()
            assert ((got - act).abs() <= dact).all(), (name, e, "act")
        y, dy = act @ down.t(), dact @ down.abs().t() + eps * ((act.abs() + dact) @ down.abs().t())
        got = taps["expert_out"][rows, torch.from_numpy(slot[r0:r1].astype(np.int64)).cuda()]
        assert ((got.double() - y).abs() <= dy).all(), (name, e, "expert_out")
    mix = (w.double().unsqueeze(2) * taps["expert_out"].double()).sum(1)
    assert ((out.double() - mix).abs() <= 2.0 ** -8 * mix.abs() +
            2.0 ** -20 * (w.unsqueeze(2) * taps["expert_out"].abs()).sum(1).double() + 1e-30).all()
    bank.close()
