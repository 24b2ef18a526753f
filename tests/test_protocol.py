"""The launches of many PCG iterations, on the host: the give-up protocol of
their grid barrier (csrc/grid_barrier.h), every access a scheduling point of a
model, their choice (csrc/persist_plan.h) and their turns (csrc/grid_turn.h)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build(tmp_path_factory, name):
    out = str(tmp_path_factory.mktemp("protocol") / name)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", "-Wextra", "-Werror",
                        "-I" + os.path.join(ROOT, "graphitethree_amd", "csrc"),
                        os.path.join(ROOT, "tests", "protocol", name + ".cpp"), "-o", out],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    return out


@pytest.fixture(scope="module")
def barrier(tmp_path_factory):
    return build(tmp_path_factory, "grid_barrier")


# workgroups, barriers, polls, groups, the one that gives up in between, samples
@pytest.mark.parametrize("n,barriers,polls,groups,quitter,samples", [
    (1, 2, 1, 1, -1, 0), (2, 1, 0, 1, -1, 0), (2, 1, 2, 1, -1, 0), (2, 1, 2, 2, -1, 0),
    (2, 2, 1, 1, -1, 0), (3, 1, 0, 1, -1, 0), (3, 1, 1, 3, -1, 30000), (2, 2, 1, 2, 1, 0),
    (5, 2, 3, 2, -1, 30000), (8, 2, 8, 3, -1, 30000), (6, 2, 6, 2, 3, 30000)])
def test_all_workgroups_pass_a_barrier_or_none(barrier, n, barriers, polls, groups, quitter,
                                               samples):
    args = [str(v) for v in (n, barriers, polls, groups, quitter, samples)]
    r = subprocess.run([barrier, *args], stdout=subprocess.PIPE, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    total, passed = int(r.stdout.split()[1]), int(r.stdout.split()[3])
    assert total > 0
    assert passed == 0 if quitter >= 0 else passed > 0  # both outcomes are met
    assert n == 1 or passed < total


def test_workgroups_that_wait_for_one_another_are_resident(tmp_path_factory):
    r = subprocess.run([build(tmp_path_factory, "persist_plan")], stdout=subprocess.PIPE,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[3]) > 0


def test_turns_go_in_order_to_one_holder_at_a_time(tmp_path_factory):
    r = subprocess.run([build(tmp_path_factory, "grid_turn")], stdout=subprocess.PIPE, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout
