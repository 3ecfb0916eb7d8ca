"""The one-wave kernels of large f32-state launches (kFWave), run on small launches by lowering their
size threshold (LV_WAVE_ELEMS): sizes around the 256-element unit, the 1024 elements behind a count
slot and the 64 slots, table and inline launches, with and without a master copy, against the oracle
bit for bit (the arithmetic is the other kernels', so any difference is an addressing or count error)."""
from __future__ import annotations

import pytest
import torch

from tests.parity_util import TensorSet, group_dict, oracle_config

pytestmark = pytest.mark.gpu

EDGES = [1, 3, 255, 256, 257, 511, 1023, 1024, 1025, 64 * 256, 64 * 1024 - 1, 64 * 1024 + 1, 70_001]


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

    monkeypatch.setenv("LV_WAVE_ELEMS", "1")
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
