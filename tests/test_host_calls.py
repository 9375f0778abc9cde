"""Locks, events and staging of the host code when something fails or engines part
(host_calls.cpp: the engine and the front end on a runtime of ordinary memory, no GPU)."""
import os
import subprocess

import pytest

from harness import ROOT


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    from neo_fft3d_amd.build import CSRC, HIPCC
    d = tmp_path_factory.mktemp("host_calls")
    objs, running = [], []
    for src in (os.path.join(CSRC, "nf3d_engine.cpp"), os.path.join(CSRC, "nf3d_frontend.cpp"),
                os.path.join(ROOT, "tests", "host_calls.cpp")):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        running.append(subprocess.Popen([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-w",
                                         "-x", "hip", "-c", src, "-o", objs[-1]]))
    assert all(p.wait(300) == 0 for p in running)
    exe = str(d / "host_calls")
    subprocess.run(["g++", "-o", exe, *objs, "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("case", ["missing_frame", "frame_throws", "pinned_refused", "engines_part", "pairs", "captured_pairs"])
def test_host(program, case):
    r = subprocess.run([program, case], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
