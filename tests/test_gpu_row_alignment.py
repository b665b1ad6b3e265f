"""Input rows off 16-byte alignment, as a view into a larger tensor is: a routed
call (bf16 and split rows, with and without a shared expert) and the official
layer give bit for bit what they give for an aligned copy of the same rows, on
either side of every change of kernels."""
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


def moved(t, elements):
    """t at `elements` past an aligned address, inside a buffer 64 elements larger."""
    buf = torch.zeros(t.numel() + 64, dtype=t.dtype, device="cuda:0")
    v = buf[elements:elements + t.numel()].view(t.shape)
    v.copy_(t)
    assert v.data_ptr() % 16
    return v


@pytest.mark.parametrize("T", [3, 5, 16, 17, 64, 130, 256, 460])
@pytest.mark.parametrize("shared", [0, 512], ids=["routed", "shared"])
@pytest.mark.parametrize("split_in", [False, True], ids=["bf16", "split_input"])
def test_routed_rows(hip, T, shared, split_in):
    k3x, ctx = hip
    H, I, E, K = 512, 512, 8, 2
    print(f"[gpu-test] rows off alignment T={T} shared={shared} split input {split_in}", flush=True)
    sys.stdout.flush()
    bank = k3x.Bank(ctx, k3x.LayerShape(H, I, E, shared))
    bank.fill_synthetic(9, 119, 123)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(T)
    x = torch.randn((T, H * (2 if split_in else 1)), device="cuda:0", generator=g).bfloat16()
    if split_in:
        x[:, H:] *= 2.0 ** -9
    ids = torch.rand((T, E), device="cuda:0", generator=g).argsort(1)[:, :K].int().contiguous()
    w = torch.rand((T, K), device="cuda:0", generator=g) + 0.1
    p = k3x.make_params(T, K, flags=k3x.FLAG_SPLIT_INPUT if split_in else 0)

    def run(rows):
        out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
        seen = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
        k3x.check(k3x.moe_forward_routed(ctx, bank, p, rows, ids, w, out,
                                         taps=dict(normed_x=seen)), "forward")
        k3x.check(ctx.synchronize(), "synchronize")
        assert torch.equal(seen, x[:, :H])
        return out

    want = run(x)
    for elements in (1, 2, 4):  # 2, 4 and 8 bytes
        assert torch.equal(run(moved(x, elements)), want), elements
    bank.close()


@pytest.mark.parametrize("T", [3, 16, 17, 40, 300])
def test_official_hidden(hip, T):
    k3x, ctx = hip
    H, L, I, Is, E, K = 1024, 512, 512, 512, 16, 2
    print(f"[gpu-test] official hidden off alignment T={T}", flush=True)
    sys.stdout.flush()
    bank = k3x.Bank(ctx, k3x.LayerShape(L, I, E, 0))
    bank.fill_synthetic(3, 119, 123)
    off = k3x.Official(ctx, bank, H, Is)
    off.fill_synthetic(4)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(T)
    hidden = torch.randn((T, H), device="cuda:0", generator=g).bfloat16()
    prefix = torch.randn((T, H), device="cuda:0", generator=g)
    ids = torch.rand((T, E), device="cuda:0", generator=g).argsort(1)[:, :K].int().contiguous()
    w = torch.rand((T, K), device="cuda:0", generator=g) + 0.1
    p = k3x.make_params(T, K, 1.0, 1e-5, k3x.GLU_SITU, 4.0, 25.0, k3x.RENORM_DOUBLE)

    def run(rows):
        out = torch.empty((T, H), dtype=torch.bfloat16, device="cuda:0")
        k3x.check(off.ffn(p, rows, prefix, out, ids, w), "ffn")
        k3x.check(ctx.synchronize(), "synchronize")
        return out

    want = run(hidden)
    for elements in (1, 2, 4):
        assert torch.equal(run(moved(hidden, elements)), want), elements
    off.close()
    bank.close()
