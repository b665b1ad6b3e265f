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
                 "scaled", "few", "wide")
        text = "\n".join(" ".join(str(int(dict(BASE, **c)[f])) for f in order) for c in calls)
        return subprocess.run([exe], input=text, capture_output=True, text=True, check=True,
                              timeout=60).stdout.split()
    return kinds


BASE = dict(hidden=7168, inter=2048, experts=384, tokens=64, top_k=16, split_act=0, split_in=0,
            scaled=0, few=0, wide=0)


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
