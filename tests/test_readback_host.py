"""Image readback's host side (csrc/readback.cpp) on a HIP stub: sizes around its chunks and limits, every call
that can fail, threads that cannot be had, other work on the device, and what a first large copy allocates."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "metal-vibe-tracer_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
MB = 1 << 20


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("readback") / "readback_host")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", CSRC,
                    "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "readback_host.cpp"),
                    os.path.join(CSRC, "readback.cpp"), "-o", out, "-ldl", "-lpthread"], check=True)
    return out


def _run(program, mode):
    r = subprocess.run([program, mode], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    line = re.compile(r"(.*) (\d+): ok staged (\d+) direct (\d+) pinned (\d+) streams (\d+)")
    return [(m[1], *map(int, m.groups()[1:])) for m in map(line.match, r.stdout.splitlines())]


def test_sizes(program):
    for _, n, staged, direct, pinned, streams in _run(program, "sizes"):
        assert (staged, direct) == ((n, 0) if n >= 8 * MB else (0, n))
        # What a first copy sets up is paid in the call itself: no stream (3 ms), little pinned memory (its first
        # use costs 0.1 ms a MB).
        assert streams == 0 and pinned <= 4 * MB


def test_known_destination(program):
    assert _run(program, "known") == [("known", 20 * MB, 0, 20 * MB, 0, 0)]


@pytest.mark.parametrize("mode", ["failures", "threads", "memory"])
def test_failures(program, mode):
    assert _run(program, mode)


def test_other_work_in_between(program):
    # A chunk that waits long shares the stream with other work: at most one chunk of each thread is staged.
    (_, n, staged, direct, _, _), = _run(program, "busy")
    assert staged + direct == n and 0 < staged <= 4 * MB
