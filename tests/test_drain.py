"""Large results drained by several threads (sbp_xfer.hpp), run on the host
against a stand-in of the runtime calls (tests/host): every way a call can meet
a lack of something ends with the whole result, as one copy call gave it."""
import os
import subprocess

import pytest

from problems_helper import ROOT


@pytest.fixture(scope="module")
def drain(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("drain") / "drain")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", os.path.join(ROOT, "tests", "host"), "-I",
                    os.path.join(ROOT, "hpc-reading-course_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "drain.cpp"), "-o", exe], check=True)

    def run(case):
        r = subprocess.run([exe, case], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
        return r.returncode, r.stdout.strip()

    return run


def test_result_is_whole(drain):
    assert drain("plain") == (0, "ok")


def test_threads_that_cannot_be_allocated(drain):
    """An exception of any kind while a thread is started must not reach the C
    entry, nor leave started threads behind unjoined."""
    assert drain("no-memory") == (0, "ok")


def test_result_of_another_device(drain):
    """A context made on one device, read by a thread whose current device is
    another (a thread's first device is 0): copy calls take the stream's."""
    assert drain("other-device") == (0, "ok")


@pytest.mark.parametrize("case", ["no-pinned", "one-pinned"])
def test_pinned_memory_that_cannot_be_allocated(drain, case):
    """The chunks are a means of speed: without them the copy call remains, and
    the failed allocation is not reported by a later call."""
    assert drain(case) == (0, "ok")
