"""How the two lanes of a recorded program meet, on modelled hardware queues (CPU only): tests/host/lanes_model.cc is built
with the product's context.cc and lanes.hip and stands in for the HIP runtime."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_lanes_on_modelled_queues(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    objs = []
    csrc = os.path.join(ROOT, "sirius_amd", "csrc")
    for src in (os.path.join(csrc, "context.cc"), os.path.join(csrc, "lanes.hip"), os.path.join(ROOT, "tests", "host", "lanes_model.cc")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        # (lanes.hip with its device code, which its registration at program start refers to)
        only = [] if src.endswith(".hip") else ["--offload-host-only"]
        built = subprocess.run([hipcc, "-std=c++17", "-O1", "-x", "hip", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                                "-packed-fp32-ops"] + only + ["-fPIC", "-c", src, "-o", objs[-1]], stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
        assert built.returncode == 0, built.stdout.decode()[-3000:]
    exe = str(tmp_path / "lanes_model")
    link = subprocess.run(["g++"] + objs + ["-o", exe, "-lpthread"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    assert link.returncode == 0, link.stdout.decode()[-3000:]
    run = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=120)
    assert run.returncode == 0, run.stdout.decode()[-4000:]
    assert " 0 failures" in run.stdout.decode()
