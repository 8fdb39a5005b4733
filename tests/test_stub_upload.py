"""Graph::gather behind a load that failed, on a stub of the device (tests/stub_upload.cpp)."""
import os
import subprocess

from tests.conftest import ROOT


def test_a_lookup_behind_a_failed_load_reads_the_ids_of_the_hosts_copy(tmp_path):
    # never those of an earlier load, nor what the memory held, which the vocabulary check has not seen
    exe = str(tmp_path / "stub_upload")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-no-pie", "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "stub_upload.cpp"),
                           os.path.join(ROOT, "eisen_amd", "csrc", "host", "graph.cpp"), "-Wl,--unresolved-symbols=ignore-all", "-Wl,-z,lazy", "-o", exe])
    done = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr
