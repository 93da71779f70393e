"""Staged host-to-device copies and the marks that order later uses after them
(tests/stage_check.cpp, over imitated streams; CPU only): several threads,
streams that begin a capture or are destroyed after their copy, replays of
captured graphs on other streams, and more copies in flight than the ring holds."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("stage") / "stage_check"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cmd = ["g++", "-O1", "-g", "-std=c++17", "-pthread", f"-I{rocm}/include",
           "-D__HIP_PLATFORM_AMD__", f"-I{os.path.join(ROOT, 'tyxonq_amd', 'csrc')}",
           os.path.join(HERE, "stage_check.cpp"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("scenario", ["two_threads", "updater_under_capture",
                                      "capture_on_own_stream", "update_after_capture",
                                      "ring_capture", "ring_gone", "in_flight", "thread_ends",
                                      "two_devices", "refused"])
def test_staging(checker, scenario):
    r = subprocess.run([str(checker), scenario], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
