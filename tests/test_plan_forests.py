"""Forests at the edges of the launch plans and of the forms beside them open and pack (no GPU: planner and packer alone)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "treebeard_amd", "csrc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("plan_forests") / "plan_forests")
    built = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-I", CSRC,
                            os.path.join(HERE, "native", "plan_forests.cpp")] +
                           [os.path.join(CSRC, s) for s in ("forest.cpp", "packer.cpp", "tuner.cpp")] + ["-o", exe], capture_output=True, text=True)
    if built.returncode != 0 and "sanitize" in built.stderr:
        pytest.skip("this g++ has no sanitizer runtime")
    assert built.returncode == 0, built.stderr[-3000:]
    return exe


def run(driver, name):
    done = subprocess.run([driver, name], capture_output=True, text=True, timeout=600)
    assert done.returncode == 0 and done.stdout.strip().endswith("ok"), (done.stdout + done.stderr)[-4000:]


def test_big_trees_open_with_every_batch(driver):
    run(driver, "big_trees")


def test_deep_forests_up_to_the_last_tail_node(driver):
    run(driver, "tail_limit")


def test_deep_trees_with_nodes_no_walk_reaches(driver):
    run(driver, "unreachable_nodes")


def test_splits_no_walk_reaches_are_no_thresholds(driver):
    run(driver, "unreachable_splits")


def test_small_forests_with_peeled_walks(driver):
    run(driver, "small_peeled")


def test_block_shapes_of_small_batches(driver):
    run(driver, "small_batches")


def test_two_trees_side_by_side_of_classifiers(driver):
    run(driver, "two_trees_of_classes")


def test_two_trees_side_by_side_of_sliced_forests(driver):
    run(driver, "two_trees_of_slices")


def test_as_many_features_as_can_be_counted(driver):
    run(driver, "most_features")


def test_room_that_own_classes_leave(driver):
    run(driver, "room_of_own_classes")


def test_plans_of_peeled_walks(driver):
    run(driver, "plans_of_peeled_walks")
