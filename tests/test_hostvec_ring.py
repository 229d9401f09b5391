"""The pinned ring of the host vectors, on the CPU: its source built against a
small runtime whose streams run nothing before they are waited for and whose
events belong to one device, with the library on one device and moved between
two by mf_init."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def ring(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ring") / "ring")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-x", "c++", "-I", os.path.join(HERE, "c", "fake_hip"),
                        os.path.join(HERE, "c", "hostvec_ring.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("devices", [1, 2])
def test_vectors_arrive(ring, devices):
    r = subprocess.run([ring] + ["2"] * (devices > 1), capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
