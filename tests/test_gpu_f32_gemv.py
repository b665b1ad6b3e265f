"""The vector form of the fp32 products (latent.hip) at its edges: odd row
counts, columns short of, at and past the staged 1024, one token to more than
a pass of eight; against float64 rounded once.  Sums are formed in double, so
every output is within one fp32 ulp (2^-23 of its value at most, plus 2^-40 of
sum |w x| where the terms cancel)."""
from __future__ import annotations

import sys

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


def rand(g, *shape):
    return torch.randn(shape, device="cuda:0", generator=g)


@pytest.mark.parametrize("rows,cols", [(1, 4), (2, 1020), (37, 1024), (129, 1028), (8, 3072)])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 8, 9, 17])
def test_matvec_edges(hip, rows, cols, T):
    k3x, ctx = hip
    print(f"[gpu-test] f32 gemv rows={rows} cols={cols} T={T}", flush=True)
    sys.stdout.flush()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(rows * cols + T)
    W, x = rand(g, rows, cols), rand(g, T, cols)
    y = torch.full((T, rows), float("nan"), device="cuda:0")
    k3x.check(k3x.dense_f32_matvec(ctx, W, x, y), "matvec")
    k3x.check(ctx.synchronize(), "synchronize")
    want = x.double() @ W.double().t()
    bound = 2.0 ** -23 * want.abs() + 2.0 ** -40 * (x.double().abs() @ W.double().abs().t())
    assert ((y.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("T", [1, 4, 7])
def test_situ_mlp_odd_rows(hip, T):
    """An odd number of gate / up pairs and of output rows.  expf and tanhf
    are about an ulp off each: 2^-20 of the activation covers them."""
    k3x, ctx = hip
    H, I, O = 1028, 36, 35
    g = torch.Generator(device="cuda:0")
    g.manual_seed(T)
    gate, up, down = rand(g, I, H) * 0.05, rand(g, I, H) * 0.05, rand(g, O, I) * 0.2
    x = rand(g, T, H)
    act, y = torch.empty((T, I), device="cuda:0"), torch.empty((T, O), device="cuda:0")
    k3x.check(k3x.dense_situ_mlp(ctx, gate, up, down, x, act, y, 4.0, 25.0), "mlp")
    k3x.check(ctx.synchronize(), "synchronize")
    gv, uv = x.double() @ gate.double().t(), x.double() @ up.double().t()
    want = 4 * torch.tanh(gv / 4) / (1 + torch.exp(-gv)) * 25 * torch.tanh(uv / 25)
    assert ((act.double() - want).abs() <= 2.0 ** -20 * want.abs() + 1e-9).all()
    out = act.double() @ down.double().t()
    assert ((y.double() - out).abs() <= 2.0 ** -23 * out.abs() +
            2.0 ** -40 * (act.double().abs() @ down.double().abs().t())).all()
