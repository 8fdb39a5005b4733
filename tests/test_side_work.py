"""Graph::run_beside on a stub of the device (tests/stub_device.cpp): whatever the device answers at each fork, the same gradients."""
import itertools
import os
import subprocess

import pytest

from tests.conftest import ROOT


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("stub") / "stub_device")
    # the entry points that the stub leaves out belong to operators that it does not run
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-no-pie", "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "stub_device.cpp"),
                           os.path.join(ROOT, "eisen_amd", "csrc", "host", "graph.cpp"), "-Wl,--unresolved-symbols=ignore-all", "-Wl,-z,lazy", "-o", exe])
    return exe


@pytest.mark.parametrize("answers", ["".join(a) for a in itertools.product("10", repeat=4)])
def test_weight_used_twice_has_the_same_gradient_whenever_the_device_catches_up(stub, answers):
    done = subprocess.run([stub, answers], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr


@pytest.mark.parametrize("answers", ["".join(a) for a in itertools.product("10", repeat=2)])
def test_products_left_for_the_pass_stay_off_the_side_stream(stub, answers):
    # a weight whose second product runs beside the chain must not take the other weights' products there with it
    done = subprocess.run([stub, "rows_of_two_lengths", answers], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr


def test_weight_of_the_feed_forward_tail_used_again_waits_for_the_side_stream(stub):
    done = subprocess.run([stub, "tail_and_its_residual", ""], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr


def test_a_window_keeps_the_operands_of_its_own_products_only(stub):
    # those that the pass's launch has read go back with the pass
    done = subprocess.run([stub, "window_with_a_narrow_layer", ""], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr


def test_products_kept_to_the_tape_run_at_their_nodes(stub):
    # and have the bits of those that the pass leaves
    done = subprocess.run([stub, "order_of_products", ""], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr


def test_products_left_by_a_pass_that_threw(stub):
    # a gradient read, cleared or left alone behind it is that of products formed at their nodes
    done = subprocess.run([stub, "pass_that_threw", ""], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr
