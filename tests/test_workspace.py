"""The prompt GEMM's per-call workspaces (csrc/qm_workspace.hip, host code): compiled against a HIP runtime on paper
(fake_hip_workspace.cpp) whose memory and events are plain counters."""
import os
import subprocess

import pytest

from arcinfer_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.path.dirname(os.path.dirname(build.HIPCC))


@pytest.fixture(scope="module")
def scenario(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ws") / "ws")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", build.CSRC, "-x", "c++",
                    os.path.join(build.CSRC, "qm_workspace.hip"), os.path.join(HERE, "fake_hip_workspace.cpp"), "-o", exe], check=True)
    return lambda name: [int(v) for v in subprocess.run([exe, name], check=True, capture_output=True, text=True).stdout.split()]


def test_what_a_call_must_have_is_enough(scenario):
    """24 MiB free, 20 needed, 30 more wanted: the call gets its 20 (without the rest) and leaves no error behind."""
    assert scenario("need_alone") == [1, 0, 0]


def test_no_stream_waits_for_another(scenario):
    """Twelve streams, eight kept buffers: a stream waits for its own last call only, the other four have the pool's memory, and a
    buffer whose work has ended serves any stream without a new allocation."""
    assert scenario("streams") == [1, 0, 8, 0, 0]


def test_small_buffers_make_room(scenario):
    """Eight small buffers don't send every larger call to the pool: it takes the place of one, once, and stays."""
    assert scenario("grow") == [1, 1, 8, 1, 8]


def test_given_back_to_the_device(scenario):
    """What is given back leaves the pool too (32 MiB stay: the buffer of the call that is enqueueing), and the next call goes on."""
    assert scenario("give_back") == [1, 1, 32, 1, 32, 0]


def test_shared_array_is_used_in_turn(scenario):
    """Four uses from two streams: each but the first waits on the GPU for the one before."""
    assert scenario("shared") == [1, 3]
