"""How the launches of f32 attention are laid out (eisen_amd/csrc/attention_f32_plan.h)."""
import os
import random
import subprocess

import pytest

from tests.conftest import ROOT

MAIN = """
#include <cstdio>
#include "attention_f32_plan.h"
int main() {
    int k8, B, S, Hq, Hkv;
    while (std::scanf("%d %d %d %d %d", &k8, &B, &S, &Hq, &Hkv) == 5) {
        const F32AttnPlan p = f32_attn_plan(k8, B, S, Hq, Hkv);
        std::printf("%lld %lld %lld %d %d %zu %zu %zu %zu %d\\n", p.qblocks, p.kblocks, p.dq_groups, p.wq, p.wk, p.fwd_lds, p.dq_lds, p.dkv_lds, p.bwd_lds, (int)p.one);
    }
}
"""
CLASSES = (2, 4, 6, 8, 10, 12, 16)  # k8, in groups of eight columns


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    (where / "main.cpp").write_text(MAIN)
    exe = str(where / "plan")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "eisen_amd", "csrc"), str(where / "main.cpp"), "-o", exe])

    def run(sizes):
        out = subprocess.run([exe], input="\n".join(" ".join(map(str, s)) for s in sizes), capture_output=True, text=True, check=True).stdout
        names = "qblocks kblocks dq_groups wq wk fwd_lds dq_lds dkv_lds bwd_lds one".split()
        return [dict(zip(names, map(int, line.split()))) for line in out.splitlines()]

    return run


def some_sizes():
    rng = random.Random(3)
    sizes = []
    for _ in range(4000):
        hkv = rng.choice([1, 1, 2, 3, 8, 16])
        sizes.append((rng.choice(CLASSES), int(2 ** rng.uniform(0, 10)), int(2 ** rng.uniform(0, 13)), hkv * rng.choice([1, 1, 2, 3, 4, 7]), hkv))
    return sizes


def test_lds_holds_what_the_waves_write_and_nothing_for_one_wave(plans):
    sizes = some_sizes()
    for (k8, B, S, Hq, Hkv), p in zip(sizes, plans(sizes)):
        dt, tile = (k8 + 3) // 4, 16 * 64 * 4
        together = p["wk"] // p["wq"]
        assert p["wk"] == together * p["wq"] and p["wk"] <= (8 if k8 <= 4 else 4)
        assert p["fwd_lds"] == (p["wq"] - 1) * (dt * tile + 128 * 4)  # every wave but the first: O, m and l
        assert p["dq_lds"] == (p["wq"] - 1) * dt * tile
        assert p["dkv_lds"] == (0 if p["wk"] == 1 else 2 * p["wk"] * tile)  # a tile of every wave, two in turn
        assert p["bwd_lds"] >= max(together * p["dq_lds"], p["dkv_lds"]) and max(p["fwd_lds"], p["bwd_lds"]) <= 64 << 10
        assert p["qblocks"] == -(-S // 32) * Hq * B and p["kblocks"] == -(-S // 32) * Hkv * B
        assert (p["dq_groups"] - 1) * together < p["qblocks"] <= p["dq_groups"] * together
        if p["kblocks"] >= 2048:
            assert p["wq"] == p["wk"] == 1 and p["fwd_lds"] == p["bwd_lds"] == 0


def test_no_launch_of_more_threads_than_there_can_be(plans):
    # 2^32 of them; either pass of its own may still fit where both together do not
    sizes = [(2, 1 << 13, 32, 1 << 12, 1 << 12), (2, 1 << 13, 32, 1 << 11, 1 << 11), (16, 1 << 15, 64, 1000, 500), (4, 65535, 1, 1023, 1), (4, 65535, 33, 512, 512)] + some_sizes()
    both = 0
    for size, p in zip(sizes, plans(sizes)):
        alone = max(p["qblocks"] * 64 * p["wq"], p["kblocks"] * 64 * p["wk"])
        together = (p["kblocks"] + p["dq_groups"]) * 64 * p["wk"]
        assert alone < 1 << 32, size
        assert not p["one"] or together < 1 << 32, size
        both += together >= 1 << 32
    assert both >= 3


def test_two_launches_for_large_grids_of_large_heads(plans):
    def one(k8, B, S, Hq, Hkv):
        return bool(plans([(k8, B, S, Hq, Hkv)])[0]["one"])

    assert not one(16, 16, 512, 8, 8) and not one(16, 16, 256, 8, 8) and not one(16, 32, 1024, 8, 1)  # 1024 key blocks and more
    assert one(16, 1, 800, 8, 8) and one(16, 1023, 32, 8, 1) and one(12, 16, 512, 8, 8) and one(4, 512, 32, 8, 8)
