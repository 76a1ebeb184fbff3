"""What staf_compute does on the host where a GPU gives the occasion only now and then: its two host sources are compiled for
the host alone and run over a runtime of this directory (md_entry_host/fake_gpu.cpp), without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "alphanesgpu_amd", "csrc")


@pytest.fixture(scope="module")
def fake_gpu(tmp_path_factory):
    d = tmp_path_factory.mktemp("fake_gpu")
    sources = [os.path.join(CSRC, s) for s in ("staf_api.hip", "staf_runtime.hip", "staf_mlp.cpp")]
    sources.append(os.path.join(ROOT, "tests", "md_entry_host", "fake_gpu.cpp"))
    objects = [str(d / f"{i}.o") for i in range(len(sources))]
    for s, o in zip(sources, objects):
        lang = [] if s.endswith("staf_mlp.cpp") else ["-x", "hip", "--offload-host-only"]
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-Wno-unused-result", *lang, "-c", s, "-o", o])
    exe = str(d / "fake_gpu")
    # (the device code that the objects would register is not there)
    subprocess.check_call(["g++", "-no-pie", "-o", exe, *objects, "-lpthread", "-Wl,--unresolved-symbols=ignore-in-object-files"])
    return exe


def scenario(exe, name):
    r = subprocess.run([exe, os.path.join(ROOT, "tests", "golden", "model_double"), name], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "ok\n")


def test_a_call_whose_stage_cannot_be_launched_leaves_nothing_behind(fake_gpu):
    """The call's first kernel is queued and reads the pinned input; the call returns -20.  It has waited for the kernel, and
    the next call with the same types sends the order of the atoms again."""
    scenario(fake_gpu, "failed_launch")


def test_a_condition_of_a_call_is_its_own(fake_gpu):
    """Another thread's poll, which clears the words of every stream, between a call's results and its return: the call still
    reports what its kernels found."""
    scenario(fake_gpu, "other_poll")


def test_a_condition_of_another_stream_is_left_to_it(fake_gpu):
    scenario(fake_gpu, "other_stream")


def test_a_program_that_asks_for_blocking_waits_gets_them(fake_gpu):
    """hipDeviceScheduleBlockingSync: the call sleeps until its stream is through, it does not watch the flags."""
    scenario(fake_gpu, "blocking_wait")
