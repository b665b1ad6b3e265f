"""The fp32 products (latent.hip) at their edges: odd row counts, columns short of,
at and past the staged 1024 and the quarters of its tail, on either side of the
short rows' own kernel (512, 768 columns), one token to more than a pass of eight; against float64 rounded once.  Sums are formed in double, so
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


@pytest.mark.parametrize("rows,cols", [(1, 4), (2, 1020), (37, 1024), (129, 1028), (8, 3072), (5, 512), (7, 516),
                                       (9, 768), (6, 772), (3, 1280), (11, 1796)])
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
    if T == 4:
        H, I = 260, 772  # gate and up a row a wave, down in the vector form
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


WEIGHTS = ("routed_down", "routed_up", "shared_gate", "shared_up", "shared_down")


@pytest.mark.parametrize("T", [1, 3])
@pytest.mark.parametrize("off", [(), ("routed_down",), ("routed_up",), ("shared_gate",),
                                 ("shared_up",), ("shared_down",), WEIGHTS],
                         ids=lambda o: "all" if len(o) > 1 else o[0] if o else "none")
def test_latent_layer_matrices_off_alignment(hip, off, T):
    """The latent layer with matrices 4 bytes past 16-byte alignment: only the
    products concerned leave the vector form (one launch more each, two with
    every matrix off; a pair off, as gate and up, is one product), and the
    results are the aligned call's within one fp32 ulp where sums are formed
    in another order (2^-22 of the value; 2^-20 of the row's largest covers what
    an ulp of the latent or of the activation moves)."""
    k3x, ctx = hip
    H, L, S, E, K, I = 132, 256, 68, 4, 2, 128
    print(f"[gpu-test] latent layer, off alignment: {off} T={T}", flush=True)
    sys.stdout.flush()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(T)
    bank = k3x.Bank(ctx, k3x.LayerShape(L, I, E, 0))
    bank.fill_synthetic(5, 119, 123)
    shapes = dict(routed_down=(L, H), routed_up=(H, L), shared_gate=(S, H), shared_up=(S, H),
                  shared_down=(H, S))
    w = {n: rand(g, *s) * 0.1 for n, s in shapes.items()}
    w["routed_norm"] = rand(g, L) * 0.1 + 1
    x = rand(g, T, H)
    ids = torch.stack([torch.randperm(E, device="cuda:0", generator=g)[:K] for _ in range(T)])
    ids = ids.int().contiguous()
    c = torch.rand((T, K), device="cuda:0", generator=g) + 0.1
    p = k3x.make_params(T, K, 1.0, 1e-6, k3x.GLU_SITU, 4.0, 25.0)

    def moved(t):
        buf = torch.empty(t.numel() + 4, device="cuda:0")
        v = buf[1:1 + t.numel()].view(t.shape)
        v.copy_(t)
        assert v.data_ptr() % 16 == 4
        return v

    def run(weights):
        out = torch.empty((T, H), device="cuda:0")
        n = ctx.stats().kernel_launches
        k3x.check(k3x.resident_moe_layer(ctx, bank, weights, p, x, ids, c, out), "latent layer")
        k3x.check(ctx.synchronize(), "synchronize")
        return out.double(), ctx.stats().kernel_launches - n

    want, n0 = run(w)
    got, n = run({m: moved(t) if m in off else t for m, t in w.items()})
    assert n - n0 == (0 if not off else 2 if len(off) > 1 else 1)
    bound = 2.0 ** -22 * want.abs() + 2.0 ** -20 * want.abs().max(1, keepdim=True).values
    assert ((got - want).abs() <= bound).all()
    bank.close()
