"""Which kernels run a call's routed experts (project-k3x_amd/csrc/k3x_select.hpp), built for the
host: sizes that no test could allocate are checked here."""
from __future__ import annotations

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def select(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("select") / "select_driver")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror",
                        f"-I{os.path.join(ROOT, 'project-k3x_amd', 'csrc')}",
                        os.path.join(ROOT, "tests", "cpp", "select_driver.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]

    def kinds(calls):
        order = ("hidden", "inter", "experts", "tokens", "top_k", "split_act", "split_in",
                 "shared", "scaled", "few", "rows", "wide")
        text = "\n".join(" ".join(str(int(dict(BASE, **c)[f])) for f in order) for c in calls)
        return subprocess.run([exe], input=text, capture_output=True, text=True, check=True,
                              timeout=60).stdout.split()
    return kinds


BASE = dict(hidden=7168, inter=2048, experts=384, tokens=64, top_k=16, split_act=0, split_in=0,
            shared=0, scaled=0, few=0, rows=0, wide=0)


@pytest.mark.parametrize("hidden,inter", [(65536, 65536), (32768, 131072), (128, 1 << 25),
                                          (1 << 25, 128), (65536, 131072), (1 << 20, 1 << 20)])
@pytest.mark.parametrize("split", [0, 1])
def test_large_experts_leave_32_bit_addressing(select, hidden, inter, split):
    """From 2^32 weights a matrix the streaming GEMM's 32-bit offsets do not
    reach an expert's tiles: such calls take the kernel with 64-bit ones."""
    calls = [dict(hidden=hidden, inter=inter, experts=1, top_k=1, tokens=t, split_act=split,
                  split_in=s) for t in (1, 4, 5, 17, 200) for s in (0, 1)]
    assert set(select(calls)) == {"narrow"}
    just_below = [dict(c, hidden=min(hidden, 16384), inter=min(inter, 131072), tokens=5)
                  for c in calls]
    assert set(select(just_below)) == {"stream"}


def test_long_activation_rows_leave_32_bit_addressing(select):
    rows = dict(hidden=8192, inter=128, experts=8, top_k=1)
    assert select([dict(rows, tokens=(1 << 18) - 1), dict(rows, tokens=1 << 18),
                   dict(rows, tokens=1 << 17, split_in=1)]) == ["stream", "narrow", "narrow"]


def test_few_pairs_keep_the_split_k_kernels(select):
    """Calls of few pairs run the decode kernels' row chunks: the streaming GEMM, which walks all
    of K in one wave, is slower there (7168 x 2048 experts, layer us row chunks / streaming: 2
    experts, 5 tokens 45 / 68; 4 experts, Top-2, 11 tokens 66 / 73)."""
    def kind(H, E, K, T, **more):
        return select([dict(hidden=H, experts=E, top_k=K, tokens=T, rows=1, **more)])[0]
    for E, K, T in ((1, 1, 5), (1, 1, 18), (1, 1, 33), (1, 1, 44), (2, 1, 30), (2, 2, 16), (2, 2, 33),
                    (4, 2, 5), (4, 2, 13), (4, 4, 8), (16, 4, 6), (64, 4, 7), (384, 4, 5)):
        assert kind(7168, E, K, T) == "rows", (E, K, T)
    for E, K, T in ((1, 1, 19), (1, 1, 32), (1, 1, 45), (3, 2, 33), (8, 2, 16), (16, 8, 5), (4, 4, 9),
                    (384, 16, 5)):
        assert kind(7168, E, K, T) == "stream", (E, K, T)
    assert kind(1024, 16, 4, 5) == "rows" and kind(1024, 16, 2, 11) == "stream"
    assert kind(1024, 1, 1, 6) == "rows" and kind(1024, 1, 1, 7) == "stream"
    assert kind(7168, 4, 2, 5, split_in=1) == "stream"
    assert select([dict(hidden=7168, experts=4, top_k=2, tokens=5)]) == ["stream"]


def test_busy_experts_take_the_wide_gemm(select):
    """From 128 tokens the choice of the wide GEMM looks at the work, not at the tokens alone:
    few experts with many rows each fill it long before 448 tokens (16 experts of 7168 x 2048,
    Top-16, 416 tokens: streaming 823 us, wide 598)."""
    def kind(H, I, E, K, T, **more):
        return select([dict(hidden=H, inter=I, experts=E, top_k=K, tokens=T, wide=1, **more)])[0]
    for H, I, E, K, T in ((7168, 2048, 16, 16, 192), (7168, 2048, 8, 8, 300), (7168, 2048, 16, 8, 331),
                          (7168, 2048, 64, 16, 256), (7168, 2048, 128, 16, 300),
                          (3584, 3072, 16, 16, 192), (3584, 3072, 8, 8, 300), (4096, 1536, 16, 16, 256),
                          (4096, 1536, 64, 16, 331), (7168, 2048, 384, 16, 448), (512, 512, 4, 1, 448)):
        assert kind(H, I, E, K, T) == "wide", (H, I, E, K, T)
    for H, I, E, K, T in ((7168, 2048, 16, 16, 128), (7168, 2048, 8, 8, 256), (7168, 2048, 16, 8, 256),
                          (7168, 2048, 4, 4, 447), (7168, 2048, 8, 8, 331), (7168, 2048, 64, 16, 160), (7168, 2048, 64, 8, 300),
                          (7168, 2048, 384, 16, 331), (3584, 3072, 896, 16, 447),
                          (4096, 1536, 16, 8, 447), (1024, 512, 64, 16, 447)):
        assert kind(H, I, E, K, T) == "stream", (H, I, E, K, T)
    assert [kind(7168, 2048, 128, 16, t, shared=1) for t in (300, 352)] == ["stream", "wide"]
    assert [kind(7168, 2048, 64, 8, t, shared=1) for t in (384, 416)] == ["stream", "wide"]
    assert kind(7168, 2048, 384, 16, 128, scaled=1) == "wide"
    assert kind(7168, 2048, 16, 16, 416, split_in=1) == "stream"
    assert select([dict(tokens=4096)]) == ["stream"]
