"""Layers past 32-bit byte offsets.

Experts of 2^32 weights a matrix: routed calls of a few tokens and of more than
one row tile, against float64 products of the bank's own dequantised rows.

The fp32 sums run over 32768 and 131072 columns of random codes, their errors
a random walk far below the bf16 rounding of the activation (2^-9 of each
value): relative error norms at most 2^-8 for the activation, and 2^-7 for the
down projection, which carries it.

Rows of 2^25 elements, 64 of which the dense projections' rows kernel cannot
address: a shared expert over 17 tokens against the same tokens in calls of
the GEMV's size (16 and 1), whose sums differ in order alone -- random walks of
2^25 fp32 terms' roundings, bf16 activations: relative error norm at most 2^-7.
"""
from __future__ import annotations

import sys

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

H, I = 32768, 131072


def test_experts_past_32_bit_offsets():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import k3x_amd as k3x
    ctx = k3x.Context(0)
    bank = k3x.Bank(ctx, k3x.LayerShape(H, I, 1, 0))
    bank.fill_synthetic(31, 119, 121)
    print(f"[gpu-test] one expert of {H} x {I}, {bank.bytes() >> 20} MiB", flush=True)
    sys.stdout.flush()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(3)
    x = (torch.randn((17, H), device="cuda:0", generator=g) / 64).bfloat16()

    def product(rows, matrix, n, step):
        """rows . (matrix, n rows)^T in float64, `step` matrix rows at a time."""
        return torch.cat([rows.double() @ bank.dequant_rows(0, matrix, r, step).double().t()
                          for r in range(0, n, step)], 1)

    gate, up = product(x, 0, I, 4096), product(x, 1, I, 4096)
    act = gate / (1 + torch.exp(-gate)) * up
    for T in (3, 5, 17):
        print(f"[gpu-test] large experts T={T}", flush=True)
        out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
        taps = dict(act=torch.empty((T, I), dtype=torch.bfloat16, device="cuda:0"),
                    expert_out=torch.empty((T, 1, H), device="cuda:0"))
        ids = torch.zeros((T, 1), dtype=torch.int32, device="cuda:0")
        w = torch.ones((T, 1), device="cuda:0")
        k3x.check(k3x.moe_forward_routed(ctx, bank, k3x.make_params(T, 1), x[:T].contiguous(),
                                         ids, w, out, taps=taps), "forward")
        k3x.check(ctx.synchronize(), "synchronize")
        got = taps["act"].double()
        rel = ((got - act[:T]).norm(dim=1) / act[:T].norm(dim=1)).max()
        assert rel <= 2.0 ** -8, (T, float(rel))
        y = product(taps["act"], 2, H, 1024)
        rel = ((taps["expert_out"][:, 0].double() - y).norm(dim=1) / y.norm(dim=1)).max()
        assert rel <= 2.0 ** -7, (T, float(rel))
        rel = ((out.double() - y).norm(dim=1) / y.norm(dim=1)).max()
        assert rel <= 2.0 ** -7, (T, float(rel))
    bank.close()
    ctx.close()


def test_shared_expert_of_rows_past_32_bit_offsets():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import k3x_amd as k3x
    ctx = k3x.Context(0)
    H, S, T = 1 << 25, 128, 17
    bank = k3x.Bank(ctx, k3x.LayerShape(H, 128, 1, S))
    bank.fill_synthetic(32, 119, 120, shared_sigma=0.02)
    print(f"[gpu-test] shared expert of {H} columns, {bank.bytes() >> 20} MiB", flush=True)
    sys.stdout.flush()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(4)
    x = (torch.randn((T, H), device="cuda:0", generator=g) / 64).bfloat16()

    def run(a, b):
        n = b - a
        print(f"[gpu-test] long rows, tokens {a} to {b}", flush=True)
        out = torch.empty((n, H), dtype=torch.bfloat16, device="cuda:0")
        taps = dict(shared_act=torch.empty((n, S), dtype=torch.bfloat16, device="cuda:0"),
                    shared_out=torch.empty((n, H), device="cuda:0"))
        k3x.check(k3x.moe_forward_routed(ctx, bank, k3x.make_params(n, 1), x[a:b],
                                         torch.zeros((n, 1), dtype=torch.int32, device="cuda:0"),
                                         torch.ones((n, 1), device="cuda:0"), out, taps=taps),
                  "forward")
        k3x.check(ctx.synchronize(), "synchronize")
        return taps["shared_act"].double(), taps["shared_out"]

    act, y = run(0, T)
    parts = [run(0, 16), run(16, T)]
    want_act, want = (torch.cat([p[i] for p in parts]) for i in range(2))
    assert float(want_act.abs().min()) > 0 and float(want_act.abs().max()) < 1e4
    assert float((act - want_act).norm() / want_act.norm()) <= 2.0 ** -7
    assert float((y - want).norm() / want.norm()) <= 2.0 ** -7
    bank.close()
    ctx.close()
