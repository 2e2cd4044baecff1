"""What an ensemble does as the device memory gets short (host code on the CPU,
against a stand-in of the HIP runtime): it steps with the stored-q schedule
where there is room for the members' second accumulators, and is made without
them where there is not."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "solar_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")

# per stage: its number, the q and the qw buffer it reads, stored q or all
STORED_Q = "000q 100q 211q 311q 400q"
STORE_ALL = "000a 110a 200a 310a 400a"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("ensemble") / "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC, "-I",
                    NATIVE, os.path.join(NATIVE, "ensemble_check.cpp")]
                   + [os.path.join(CSRC, f) for f in ("solar_ensemble.cpp", "solar_tables.cpp", "solar_hostcopy.cpp")]
                   + ["-pthread", "-o", out], check=True)
    return out


def _run(program, *states, **env):
    env = dict({k: v for k, v in os.environ.items() if k != "SOLAR_STEP_STORE_ALL"}, **env)
    r = subprocess.run([program, *map(str, states)], capture_output=True, text=True, timeout=60, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    order, held = r.stdout.strip().splitlines()[-1].split(",")
    return order.split(), int(held)


# two states, one accumulator, ghosts and edge columns of these members take 3.4 states' worth
@pytest.mark.parametrize("states,order,held", [(3.5, STORE_ALL, 3), (4.5, STORE_ALL, 3), (5.3, STORE_ALL, 3),
                                               (5.5, STORED_Q, 4), (40, STORED_Q, 4)])
def test_schedule_by_the_memory_there_is(program, states, order, held):
    got, have = _run(program, states)
    assert list(dict.fromkeys(got)) == order.split()
    assert have == held


def test_the_switch_declines_the_second_accumulator(program):
    got, have = _run(program, 40, SOLAR_STEP_STORE_ALL="1")
    assert list(dict.fromkeys(got)) == STORE_ALL.split() and have == 3


# memory that is free, but not in pieces: the second member's accumulator fails (3.5, 3.8), its
# ghosts do (4.3); the first member's state is a bit less than half of the two
@pytest.mark.parametrize("states", [3.5, 3.8, 4.3])
def test_accumulators_that_fail_on_the_way_are_given_back(program, states):
    got, have = _run(program, states, 40)
    assert list(dict.fromkeys(got)) == STORE_ALL.split() and have == 3


def test_too_little_memory_is_an_error(program):
    r = subprocess.run([program, "3.2"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 1 and "hipMalloc" in r.stdout
