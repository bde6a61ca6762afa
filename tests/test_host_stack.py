"""Stack frames of the engine's host code: its entry points are called from threads that
may have a small stack (bar: 16 KB a frame)."""
import os
import subprocess

import pytest

from mpsqmc_amd import build as B


def test_frames_are_small(tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    obj = str(tmp_path / "engine.o")
    flags = [f for f in B.HIPCC_FLAGS if f != "-shared"]
    subprocess.check_call([hipcc, *flags, "--cuda-host-only", "-fstack-usage", "-c", "-I",
                           os.path.join(B.ROOT, "include"), "-I", B.CSRC, os.path.join(B.CSRC, "mqe_engine.hip"),
                           "-o", obj])
    frames = {}
    for line in open(str(tmp_path / "engine.su")):
        name, size = line.split("\t")[:2]
        frames[name.split(":")[-1]] = int(size)
    assert any("overlaps_in_workspace" in f for f in frames)
    big = {f: n for f, n in frames.items() if n > 16384}
    assert not big, big
