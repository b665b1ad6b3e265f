"""The dense projections at the edges of the rows kernel's token tiles
(pipeline.hip, dense_rows_kernel), and on either side of the GEMV's and the
wide GEMM's ranges (the wide GEMM's split kernels among them).

* The layer's shared expert against float64, element-wise: the projections'
  fp32 sums within 2^-16 sum |w x| (at most 2304 terms of 2^-24, several times
  over), the SwiGLU activation rounded to bf16 (2^-8).
* The official layer's projections (bf16 latent, split activations, fp32
  routed and shared rows, the output formula): a batch against the same
  tokens run at most 16 at a time on the GEMVs.  The latent differs by one
  bf16 ulp at most beyond what the two fp32 sums differ by (each within 2^-16
  sum |w x| <= 2^-16 |w| |x| of the exact one; |w| <= 1.5 * 0.02 sqrt(H) for
  the synthetic rows), which shows where a sum cancels to near zero; what that
  moves downstream is a rounding here and there, below 2^-7 in relative error
  norm as for the layer's other kernels.
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


def say(msg):
    print(f"[gpu-test] {msg}", flush=True)
    sys.stdout.flush()


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("H,S", [(640, 384), (2304, 128)], ids=["few_tiles", "more_tiles_than_waves"])
@pytest.mark.parametrize("T", [5, 16, 17, 32, 33, 64, 65, 127, 128, 193, 255, 256])
@pytest.mark.parametrize("split_in", [False, True], ids=["bf16", "split_input"])
def test_shared_expert_rows(hip, H, S, T, split_in):
    k3x, ctx = hip
    say(f"shared expert H={H} S={S} T={T} split input {split_in}")
    g = torch.Generator(device="cuda:0")
    g.manual_seed(T + H)
    bank = k3x.Bank(ctx, k3x.LayerShape(H, 128, 4, S))
    bank.fill_synthetic(7, 119, 123)
    mats = [torch.randn(s, device="cuda:0", generator=g).mul_(0.05).bfloat16()
            for s in ((S, H), (S, H), (H, S))]
    assert bank.upload_shared(*[bits(m) for m in mats]) == 0
    gate, up, down = (m.double() for m in mats)
    x = torch.randn((T, H), device="cuda:0", generator=g)
    hi = x.bfloat16()
    xin, xv = hi, hi.double()
    if split_in:
        lo = (x - hi.float()).bfloat16()
        xin, xv = torch.cat([hi, lo], 1).contiguous(), hi.double() + lo.double()
    ids = (torch.arange(T, device="cuda:0") % 4).int().view(T, 1).contiguous()
    w = torch.ones((T, 1), device="cuda:0")
    out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
    taps = dict(shared_act=torch.empty((T, S), dtype=torch.bfloat16, device="cuda:0"),
                shared_out=torch.empty((T, H), device="cuda:0"))
    params = k3x.make_params(T, 1, flags=k3x.FLAG_SPLIT_INPUT if split_in else 0)
    k3x.check(k3x.moe_forward_routed(ctx, bank, params, xin, ids, w, out, taps=taps), "forward")
    k3x.check(ctx.synchronize(), "synchronize")
    eps = 2.0 ** -16
    gv, uv = xv @ gate.t(), xv @ up.t()
    dg, du = eps * (xv.abs() @ gate.abs().t()), eps * (xv.abs() @ up.abs().t())
    silu = gv / (1 + torch.exp(-gv))
    act = silu * uv
    dact = 1.1 * (uv.abs() * dg + silu.abs() * du + dg * du) + 2.0 ** -8 * act.abs() + 1e-30
    got = taps["shared_act"].double()
    assert ((got - act).abs() <= dact).all()
    y = got @ down.t()  # on the kernel's own activations
    dy = eps * (got.abs() @ down.abs().t()) + 1e-30
    assert ((taps["shared_out"].double() - y).abs() <= dy).all()
    bank.close()


# Shapes (H, L, I, Is, E, K): the second one's projections take the wide GEMM
# from 256 tokens, and its experts the wide GEMM's split class kernels from 448
# (at 460: chunks of 128 rows and last ones of 65 to 128).
ROWS, WIDE = (1024, 2304, 128, 384, 8, 2), (1024, 512, 512, 512, 16, 8)


@pytest.mark.parametrize("shape,T", [(ROWS, T) for T in (17, 32, 33, 64, 65, 100, 129, 200, 255)] +
                         [(WIDE, T) for T in (17, 255, 256, 300, 460)],
                         ids=lambda v: None if isinstance(v, int) else "rows" if v is ROWS else "wide")
def test_official_rows_match_gemv(hip, shape, T):
    k3x, ctx = hip
    H, L, I, Is, E, K = shape
    say(f"official rows {shape} T={T}")
    bank = k3x.Bank(ctx, k3x.LayerShape(L, I, E, 0))
    bank.fill_synthetic(3, 119, 123)
    off = k3x.Official(ctx, bank, H, Is)
    off.fill_synthetic(4)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(T)
    hidden = torch.randn((T, H), device="cuda:0", generator=g).bfloat16()
    prefix = torch.randn((T, H), device="cuda:0", generator=g)
    ids = torch.stack([torch.randperm(E, device="cuda:0", generator=g)[:K] for _ in range(T)])
    ids = ids.int().contiguous()
    w = torch.rand((T, K), device="cuda:0", generator=g) + 0.1

    def run(a, b):
        n = b - a
        taps = dict(latent=torch.empty((n, L), dtype=torch.bfloat16, device="cuda:0"),
                    routed=torch.empty((n, H), device="cuda:0"),
                    shared=torch.empty((n, H), device="cuda:0"))
        out = torch.empty((n, H), dtype=torch.bfloat16, device="cuda:0")
        p = k3x.make_params(n, K, 1.0, 1e-5, k3x.GLU_SITU, 4.0, 25.0, k3x.RENORM_DOUBLE)
        k3x.check(off.ffn(p, hidden[a:b], prefix[a:b], out, ids[a:b].contiguous(),
                          w[a:b].contiguous(), taps), "ffn")
        k3x.check(ctx.synchronize(), "synchronize")
        return dict(taps, out=out)

    batch = run(0, T)
    parts = [run(a, min(a + 16, T)) for a in range(0, T, 16)]
    for name, got in batch.items():
        want = torch.cat([p[name] for p in parts]).double()
        got = got.double()
        rel = float((got - want).norm() / want.norm())
        assert rel <= 2.0 ** -7, (name, rel)
        if name == "latent":
            sums = 2 * 2.0 ** -16 * 1.5 * 0.02 * H ** 0.5 * hidden.double().norm(dim=1, keepdim=True)
            assert ((got - want).abs() <= 2.0 ** -7 * want.abs() + sums).all()
    off.close()
    bank.close()
