"""The library's host code on the CPU, against a stand-in for the HIP runtime (host_runtime.cpp): what it
queues, and how it fails."""
import os
import subprocess

import pytest

from lageunha_amd import lagpm

HERE = os.path.dirname(os.path.abspath(__file__))
LIBDIR = os.path.dirname(lagpm.LIB_PATH)


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_runtime") / "host_runtime")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(os.path.dirname(HERE), "include"), os.path.join(HERE, "host_runtime.cpp"), "-o", out,
                    "-L" + LIBDIR, "-llagpm", "-Wl,-rpath," + LIBDIR, "-Wl,-rpath-link,/opt/rocm/lib", "-pthread"], check=True)
    return out


def run(program, scenario, *args):
    r = subprocess.run([program, scenario, *map(str, args)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"exit {r.returncode}: {r.stdout}{r.stderr}"
    values = dict(line.split(" ", 1) for line in r.stdout.splitlines())
    assert values.pop("end") == "0"
    return {k: float(v) for k, v in values.items()}


def test_a_build_deeper_than_the_sorted_key_bits_sorts_again(program):
    """set_tuning puts the box's depth limit back to the full depth. The keys may have been sorted for
    a shallower tree (here by tsc after a drift), and the build reads key order to the full depth."""
    got = run(program, "resort")
    assert got == {"same_tuning": 0, "other_tuning": 1, "again": 0, "sample": 1}


def test_steps_capture_no_graph(program):
    """Whole steps queue the same kernels with set_step_graphs on and off, and capture nothing."""
    got = run(program, "steps")
    assert got.pop("captures") == 0
    assert len(got) == 3 and len(set(got.values())) == 1 and min(got.values()) > 20


def test_first_copies_of_two_threads_share_one_set_of_slots(program):
    """Two threads make a context's first large copies at once: one set of pinned slots is made for them."""
    assert run(program, "first_copies") == {"pinned": 1}


def test_large_copy_without_host_memory(program):
    """Each host allocation of a large copy fails in turn (the chunk list, the threads' states): the copy
    returns, with LAGPM_E_NOMEM or complete, and the process goes on."""
    assert run(program, "no_host_memory") == {"refused": 1, "done_some": 1, "other": 0, "partial": 0}


def test_build_times_cover_the_build_alone(program):
    """ms_build of a step is the octree build (here counted in its kernels: 3 for the nodes, one a level for the
    moments, 3 for the groups), without the sort and the PM kick, whether phase events are recorded or not."""
    got = run(program, "build_times")
    assert len(got) == 8 and len(set(got.values())) == 1 and 7 <= min(got.values()) <= 11


def test_node_arrays_that_cannot_be_grown(program):
    """The growth of the node arrays (or of the walk's descriptors) fails for lack of device memory: that
    call fails, and the calls after it launch nothing on the arrays that were given up."""
    got = run(program, "no_device_memory")
    assert got == {"grow": 1, "still_none": 1, "again": 0, "many": 1, "many_again": 0, "bad_launches": 0}
