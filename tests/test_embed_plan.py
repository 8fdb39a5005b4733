"""Where the position index of the embedding scatter puts its ids (eisen_amd/csrc/embed_plan.h)."""
import os
import subprocess

import numpy as np
import pytest

from tests.conftest import ROOT

MAIN = """
#include <cstdio>
#include "embed_plan.h"
int main() {
    for (int id = 0; id < kBuckets * kBucketSlots; id++) {
        const int bucket = scatter_bucket_of(id);
        if (scatter_bucket_id(id >> kBucketBits, bucket) != id) return 1;
        std::printf("%d\\n", bucket);
    }
}
"""
GRID = """
#include <cstdio>
#include "embed_plan.h"
int main() {
    size_t n, hidden;
    while (std::scanf("%zu %zu", &n, &hidden) == 2) {
        const ScatterRunsGrid g = scatter_runs_grid(n, hidden);
        std::printf("%zu %zu %zu %zu %d %d %d\\n", g.long_blocks, g.short_blocks, g.window, kRunBlocksMax, kRunThreads, kRunWaves, g.long_marks);
    }
}
"""


@pytest.fixture(scope="module")
def bucket(tmp_path_factory):
    where = tmp_path_factory.mktemp("embed")
    (where / "main.cpp").write_text(MAIN)
    exe = str(where / "bucket")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "eisen_amd", "csrc"), str(where / "main.cpp"), "-o", exe])
    return np.array(subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split(), np.int32)  # (fails if an id does not come back)


def test_a_bucket_has_one_id_of_every_slot(bucket):
    assert np.array_equal(np.sort(bucket.reshape(-1, 256), axis=1), np.broadcast_to(np.arange(256), (bucket.size // 256, 256)))


def test_ids_a_stride_apart_are_not_all_one_workgroups(bucket):
    # a wave places its ids one after the other: at most a sixteenth of them, or 32 (half of its lanes), are one workgroup's, for strides up to 4096
    for stride in range(1, 4097):
        ids = np.arange(0, bucket.size, stride)
        assert np.bincount(bucket[ids]).max() <= max(32, ids.size // 16), stride


def test_the_scatters_launches_cover_all_rows_and_have_no_more_threads_than_a_launch_takes(tmp_path):
    (tmp_path / "main.cpp").write_text(GRID)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "eisen_amd", "csrc"), str(tmp_path / "main.cpp"), "-o", str(tmp_path / "grid")])
    # (rows of up to 2^30 - 1 columns, and as many of them as a card's memory holds: 121 of the widest, 2^20 of 131072)
    sizes = [(1, 2), (64, 2), (65, 2), (8192, 256), (8193, 256), (32768, 1024), (1 << 20, 64), (121, (1 << 30) - 2), (1 << 20, 131072), (1, (1 << 30) - 2), (65536, 2_000_000)]
    out = subprocess.run([str(tmp_path / "grid")], input="\n".join("%d %d" % s for s in sizes), capture_output=True, text=True, check=True).stdout
    for (n, hidden), line in zip(sizes, out.splitlines()):
        long_blocks, short_blocks, window, most, threads, waves, long_marks = map(int, line.split())
        assert (min(short_blocks, most) + long_blocks) * threads < 1 << 32
        assert short_blocks * waves >= -(-n // window) * -(-hidden // 256) > (short_blocks - 1) * waves and short_blocks * waves < 1 << 31
        assert (long_blocks > 0) == (-(-n // 64) >= long_marks) and long_marks in (2, 3) and window <= 8  # (a long run needs that many multiples of 64)
