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


def test_gpu_tests_of_large_launches_reach_them(walk):
    """Every form that tests/test_gpu_large_launches.py steps takes its large-launch kernel there, so those
    tests fail to cover what they are for as soon as a rule of the dispatch moves past their sizes."""
    from luminamoon_amd.optimizer.hip_backend import BUFFER_CODES
    from tests.test_gpu_large_launches import EDGES, FORMS, LARGE

    code = {"f32": 0, "bf16": 1, "f16": 2}
    for buffer, pdt, sdt, extra in FORMS:
        for count in (len(EDGES), 60):
            sizes = [EDGES[i % len(EDGES)] for i in range(count)] + [LARGE]
            args = [BUFFER_CODES[buffer], code[pdt], code[sdt], int("master_weights" in extra), *sizes]
            res = subprocess.run([*walk, "route", *map(str, args)], capture_output=True, text=True, timeout=60)
            assert res.returncode == 0, res.stdout + res.stderr
            launches = [tuple(map(int, l.split())) for l in res.stdout.split("\n") if l]
            assert len(launches) == 1 and launches[0][0] >> 30 == 1, (buffer, pdt, sdt, extra, count, launches)
