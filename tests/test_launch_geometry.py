"""Every launch the C ABI can make, checked on the CPU against the kernel it launches.

`tests/launch_walk.hip` (host code only) stands in for the HIP runtime, loads the built library and
walks modes, dtypes, options, bounds, passes, entry points, inline, table and split launches, small
and large classes, aligned tensors and views. Each recorded launch must have the threads, work units,
count slots and options of the kernel it names, stay inside the workspace, and take a kernel's form
for large launches exactly where there is one."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    from luminamoon_amd import build_ext

    if shutil.which(build_ext.hipcc()) is None and not os.path.exists(build_ext.hipcc()):
        pytest.skip("hipcc not found")
    if not os.path.exists(build_ext.OUT):
        build_ext.build()
    exe = str(tmp_path_factory.mktemp("walk") / "launch_walk")
    cmd = [build_ext.hipcc(), f"--offload-arch={build_ext.ARCH}", "--offload-host-only", "-O1", "-std=c++17", "-rdynamic",
           "-I", os.path.join(ROOT, "include"), "-I", build_ext.CSRC, os.path.join(HERE, "launch_walk.hip"), "-o", exe, "-ldl"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    return [exe, build_ext.OUT]


def test_every_launch_has_its_kernels_geometry(walk):
    res = subprocess.run(walk, capture_output=True, text=True, timeout=600)
    print(res.stdout)
    assert res.returncode == 0, res.stdout[-4000:] + res.stderr[-1000:]
    m = re.search(r"(\d+) calls, (\d+) unit launches checked, (\d+) of large forms, (\d+) of one-wave blocks, 0 mismatches", res.stdout)
    assert m, res.stdout[-2000:]
    assert all(int(x) > 1000 for x in m.groups())  # the walk reached what it is for
