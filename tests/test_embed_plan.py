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
