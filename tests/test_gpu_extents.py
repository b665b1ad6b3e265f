"""The one-launch extent check (storage.hip) at the edges of its chunks, and
the device admission that rests on it (k3x_hip_bank_upload_expert_device).

CRCs over sizes around what the host folds itself, a lane's words, a wave's 16 KiB, a workgroup's 64 KiB
and the step to 64 KiB chunks at 32 MiB, against the oracle's CRC32C.  An
admission with one extent corrupted, or a 0xFF byte in one array of scales,
is refused with that extent's code before the slot is touched, in the order
of the extents; the next good one succeeds (the check's counters are left
clear)."""
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


@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 1008, 1023, 1024, 1025, 4079, 4080, 4095, 4096, 4097, 16384 - 16, 16384, 16384 + 16, 65536 - 16, 65536,
                               65536 + 31, 64 * 16384, 65 * 16384 + 16, (1 << 20) + 7,
                               (32 << 20) - 16, 32 << 20, (32 << 20) + 65536 + 5])
def test_crc_chunk_edges(hip, oracle, n):
    _, ctx = hip
    print(f"[gpu-test] crc chunk edge n={n}", flush=True)
    host = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8)
    dev = torch.from_numpy(host).to("cuda:0")
    st, crc = ctx.crc32c(dev, n)
    assert st == 0 and crc == oracle.crc32c(host.tobytes())


def test_crc_of_few_bytes_takes_no_launch(hip, oracle):
    """Below 1 KiB, and below 4 KiB with a tail, the bytes are copied and folded on
    the host: a launch and a second copy would take half as long again."""
    _, ctx = hip
    host = np.random.default_rng(4).integers(0, 256, 4096, dtype=np.uint8)
    dev = torch.from_numpy(host).to("cuda:0")
    for n, launches in ((100, 0), (512, 0), (1023, 0), (1024, 1), (1030, 0), (4095, 0), (4096, 1)):
        before = ctx.stats().kernel_launches
        st, crc = ctx.crc32c(dev, n)
        assert st == 0 and crc == oracle.crc32c(host[:n].tobytes()), n
        assert ctx.stats().kernel_launches - before == launches, n


def test_admission_refusals(hip, oracle):
    k3x, ctx = hip
    H, I = 384, 256
    print("[gpu-test] admission refusals", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(5)
    n = H * I

    def expert(seed):
        r = np.random.default_rng(seed)
        return [r.integers(0, 256, n // 2, dtype=np.uint8) if i % 2 == 0 else
                r.integers(119, 124, n // 32, dtype=np.uint8) for i in range(6)]

    bank, want = (k3x.Bank(ctx, k3x.LayerShape(H, I, 3, 0)) for _ in range(2))
    good, ids = expert(1), (11, 12, 13)
    crcs = [oracle.crc32c(a.tobytes()) for a in good]
    dev = lambda ex: [torch.from_numpy(a).to("cuda:0") for a in ex]  # noqa: E731
    names = ("gate_packed", "gate_scales", "up_packed", "up_scales", "down_packed", "down_scales")
    assert want.upload_expert(1, dict(zip(names, good)), ids) == 0

    def same():
        for m, rows in ((0, I), (1, I), (2, H)):
            a, b = bank.dequant_rows(1, m, 0, rows), want.dequant_rows(1, m, 0, rows)
            if not torch.equal(a.view(torch.int32), b.view(torch.int32)):
                return False
        return bank.find(12)[1:] == (1, 1)

    assert bank.upload_expert_device(1, dev(good), ids, crcs) == 0 and same()
    for i in range(6):  # one extent's CRC is another's
        ex = expert(2)
        c = [oracle.crc32c(a.tobytes()) for a in ex]
        c[i] ^= 1 << int(rng.integers(32))
        assert bank.upload_expert_device(1, dev(ex), ids, c) == (11 if i % 2 else 10), i
        assert same(), i
    for i in (1, 3, 5):  # a 0xFF scale, with and without CRCs
        ex = expert(3)
        ex[i][int(rng.integers(n // 32))] = 0xFF
        c = [oracle.crc32c(a.tobytes()) for a in ex]
        for crc in (c, None):
            assert bank.upload_expert_device(1, dev(ex), ids, crc) == k3x.ERR_INVALID_MXFP4
            assert same(), i
        # The extents' order decides which fault is named.
        late = list(c)
        late[5] ^= 1
        early = list(c)
        early[0] ^= 1
        assert bank.upload_expert_device(1, dev(ex), ids, early) == 10
        assert bank.upload_expert_device(1, dev(ex), ids, late) == \
            (11 if i == 5 else k3x.ERR_INVALID_MXFP4)
    # A code byte 0xFF is an ordinary pair of codes.
    ok = expert(4)
    ok[0][:] = 0xFF
    assert bank.upload_expert_device(0, dev(ok), (21, 22, 23), None) == 0
    assert bank.upload_expert_device(1, dev(good), ids, crcs) == 0 and same()
    bank.close()
    want.close()
