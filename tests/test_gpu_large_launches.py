"""The kernels of large launches (kFLarge), run on small launches by lowering their size threshold
(LV_LARGE_ELEMS): the one-wave kernels with f32 state, the counting pass in 4096-element units with any
state. Sizes around the 256-element unit, the 1024 elements behind a count slot, the 64 slots and the
4096-element unit, table and inline launches, with and without a master copy, against the oracle
bit for bit (the arithmetic is the other kernels', so any difference is an addressing or count error)."""
from __future__ import annotations

import pytest
import torch

from tests.parity_util import TensorSet, group_dict, oracle_config

pytestmark = pytest.mark.gpu

EDGES = [1, 3, 255, 256, 257, 511, 1023, 1024, 1025, 4095, 4097, 8192 + 2049, 64 * 256, 64 * 1024 - 1, 64 * 1024 + 1, 70_001]


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("buffer,pdt,master", [
    (2, "f32", "none"), ("T2", "f32", "none"), (1, "f32", "none"), ("T1", "f32", "none"),
    ("T2", "bf16", "none"), ("T2", "f16", "none"), ("T1", "bf16", "none"), ("T1", "f16", "none"),
    (2, "bf16", "full"), (2, "f16", "semi"), ("T2", "bf16", "full"), ("T2", "f16", "full"),
    (1, "bf16", "full"), (1, "f16", "full"), ("T1", "bf16", "semi"), ("T1", "f16", "full"),
])
def test_one_wave_launches_match_oracle(buffer, pdt, master, count, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    from luminamoon_amd.optimizer import hip_backend
    from oracle import oracle as O

    monkeypatch.setenv("LV_LARGE_ELEMS", "1")
    group = group_dict(buffer=buffer, lr=1e-3, master_weights=master)
    cfg = oracle_config(O, group)
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    host = TensorSet(sizes, pdt, pdt, "f32", buffer in (2, "T2"), master != "none", 77)
    dev = host.to("cuda")
    stepper = hip_backend.HipStepper()
    print(f"[case] one-wave {buffer} {pdt} master={master} tensors={count}", flush=True)
    for step in (1, 2, 3):
        grads = host.grads(step, 77)
        host.oracle_step(O, cfg, grads, step, threads=4)
        dev.hip_step(stepper, group, [g.cuda() for g in grads], step)
        torch.cuda.synchronize()
        host.assert_equal(dev, f"step {step}")
    assert all(int(torch.count_nonzero(ws)) == 0 for ws in stepper.workspace._bufs.values())


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("buffer,pdt,sdt,extra", [
    (1, "bf16", "f32", {}), ("T2", "f32", "f32", {}), ("T1", "f16", "f16", {"state_precision": "param"}),
    (2, "bf16", "bf16", {"state_precision": "param"}), (2, "bf16", "f32", {"master_weights": "full"}),
    ("T2", "f16", "f32", {"stochastic_rounding": False, "weight_decay": 0.0}), (1, "f32", "f32", {"bound": False}),
])
def test_two_pass_large_launches_match_oracle(buffer, pdt, sdt, extra, count, monkeypatch):
    """Counting and applying passes take units of their own kernels' sizes."""
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    from luminamoon_amd.optimizer import hip_backend
    from oracle import oracle as O

    monkeypatch.setenv("LV_LARGE_ELEMS", "1")
    group = group_dict(buffer=buffer, lr=1e-3, fused_single_pass=False, **extra)
    cfg = oracle_config(O, group)
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    host = TensorSet(sizes, pdt, pdt, sdt, buffer in (2, "T2"), "master_weights" in extra, 78)
    dev = host.to("cuda")
    stepper = hip_backend.HipStepper()
    print(f"[case] two-pass {buffer} {pdt}/{sdt} {extra} tensors={count}", flush=True)
    for step in (1, 2):
        grads = host.grads(step, 78)
        host.oracle_step(O, cfg, grads, step, threads=4)
        dev.hip_step(stepper, group, [g.cuda() for g in grads], step)
        torch.cuda.synchronize()
        host.assert_equal(dev, f"step {step}")
    assert all(int(torch.count_nonzero(ws)) == 0 for ws in stepper.workspace._bufs.values())
