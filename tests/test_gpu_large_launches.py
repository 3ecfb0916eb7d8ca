"""The kernels of large launches (kFLarge): the one-wave kernels with f32 state, the counting pass in
4096-element units with any state, optimistic lanes. A zero tensor of 2^27 elements on the device alone
makes the launch large (tests/test_launch_geometry.py checks on the CPU that it does); the small tensors
beside it are compared. Sizes around the 256-element unit, the 1024 elements behind a count slot, the 64
slots and the 4096-element unit, in table and inline launches, with and without a master copy; views,
inactive ranges, shard offsets, single passes, split launches and graph steps. Against the oracle bit for
bit (the arithmetic is the other kernels', so any difference is an addressing or count error)."""
from __future__ import annotations

import pytest
import torch

from tests.parity_util import TensorSet, group_dict, oracle_config
from tests.test_gpu_special_values import GRAD_SPECIALS, M_SPECIALS, P_SPECIALS, V_SPECIALS, _assert_same, _inject

pytestmark = pytest.mark.gpu

EDGES = [1, 3, 255, 256, 257, 511, 1023, 1024, 1025, 4095, 4097, 8192 + 2049, 64 * 256, 64 * 1024 - 1, 64 * 1024 + 1, 70_001]
# At least kLargeElems, and with 60 tensors beside it a mean tensor that one-wave table launches ask for (wave_table_mean).
LARGE = 1 << 27


def _large(host):
    """The device copy of `host` with a last tensor of LARGE zeros, and that tensor's gradient."""
    dev = host.to("cuda")
    dev.sizes = host.sizes + [LARGE]

    def zeros(like):
        return None if like[0] is None else torch.zeros(LARGE, dtype=like[0].dtype, device="cuda")

    for xs in (dev.p, dev.m, dev.v, dev.mp):
        xs.append(zeros(xs))
    dev.sc.append(torch.tensor([0, 0, 0, 1, 1, 0], dtype=torch.float32, device="cuda"))
    return dev, torch.zeros(LARGE, dtype=host.gdt, device="cuda")


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("buffer,pdt,master", [
    (2, "f32", "none"), ("T2", "f32", "none"), (1, "f32", "none"), ("T1", "f32", "none"),
    ("T2", "bf16", "none"), ("T2", "f16", "none"), ("T1", "bf16", "none"), ("T1", "f16", "none"),
    (2, "bf16", "full"), (2, "f16", "semi"), ("T2", "bf16", "full"), ("T2", "f16", "full"),
    (1, "bf16", "full"), (1, "f16", "full"), ("T1", "bf16", "semi"), ("T1", "f16", "full"),
])
def test_one_wave_launches_match_oracle(buffer, pdt, master, count):
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    from luminamoon_amd.optimizer import hip_backend
    from oracle import oracle as O

    group = group_dict(buffer=buffer, lr=1e-3, master_weights=master)
    cfg = oracle_config(O, group)
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    host = TensorSet(sizes, pdt, pdt, "f32", buffer in (2, "T2"), master != "none", 77)
    dev, fill = _large(host)
    stepper = hip_backend.HipStepper()
    print(f"[case] one-wave {buffer} {pdt} master={master} tensors={count}", flush=True)
    for step in (1, 2, 3):
        grads = host.grads(step, 77)
        host.oracle_step(O, cfg, grads, step, threads=4)
        dev.hip_step(stepper, group, [g.cuda() for g in grads] + [fill], step)
        torch.cuda.synchronize()
        host.assert_equal(dev, f"step {step}")
    assert all(int(torch.count_nonzero(ws)) == 0 for ws in stepper.workspace._bufs.values())


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("buffer,pdt,sdt,extra", [
    (1, "bf16", "f32", {}), ("T2", "f32", "f32", {}), ("T1", "f16", "f16", {"state_precision": "param"}),
    (2, "bf16", "bf16", {"state_precision": "param"}), (2, "bf16", "f32", {"master_weights": "full"}),
    ("T2", "f16", "f32", {"stochastic_rounding": False, "weight_decay": 0.0}), (1, "f32", "f32", {"bound": False}),
])
def test_two_pass_large_launches_match_oracle(buffer, pdt, sdt, extra, count):
    """Counting and applying passes take units of their own kernels' sizes."""
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    from luminamoon_amd.optimizer import hip_backend
    from oracle import oracle as O

    group = group_dict(buffer=buffer, lr=1e-3, fused_single_pass=False, **extra)
    cfg = oracle_config(O, group)
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    host = TensorSet(sizes, pdt, pdt, sdt, buffer in (2, "T2"), "master_weights" in extra, 78)
    dev, fill = _large(host)
    stepper = hip_backend.HipStepper()
    print(f"[case] two-pass {buffer} {pdt}/{sdt} {extra} tensors={count}", flush=True)
    for step in (1, 2):
        grads = host.grads(step, 78)
        host.oracle_step(O, cfg, grads, step, threads=4)
        dev.hip_step(stepper, group, [g.cuda() for g in grads] + [fill], step)
        torch.cuda.synchronize()
        host.assert_equal(dev, f"step {step}")
    assert all(int(torch.count_nonzero(ws)) == 0 for ws in stepper.workspace._bufs.values())


@pytest.mark.parametrize("sizes", [EDGES, EDGES * 3 + [70_003]], ids=["one-launch", "two-launches"])
@pytest.mark.parametrize("buffer", [2, "T2"])
def test_f32_radial_large_launches_match_oracle(buffer, sizes):
    """Block b on unit b with fewer blocks per CU; the unit records and their fold keep unit order."""
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    from luminamoon_amd.optimizer import hip_backend
    from oracle import oracle as O

    group = group_dict(buffer=buffer, lr=1e-3, bound_type="radial")
    cfg = oracle_config(O, group)
    host = TensorSet(sizes, "f32", "f32", "f32", True, False, 80)
    dev, fill = _large(host)
    stepper = hip_backend.HipStepper()
    print(f"[case] radial {buffer} tensors={len(sizes)}", flush=True)
    with O.radial_sum_f64():
        for step in (1, 2, 3):
            grads = host.grads(step, 80)
            host.oracle_step(O, cfg, grads, step, threads=4)
            dev.hip_step(stepper, group, [g.cuda() for g in grads] + [fill], step)
            torch.cuda.synchronize()
            host.assert_equal(dev, f"step {step}")
    assert all(int(torch.count_nonzero(ws)) == 0 for ws in stepper.workspace._bufs.values())


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("buffer,extra", [
    (1, {}), (2, {}), ("T1", {}), ("T2", {}), (2, {"cautious": False}), ("T1", {"fused_single_pass": False}),
])
def test_f32_params_with_separate_masters_match_oracle(buffer, extra, count):
    """An f32 param whose master copy is another buffer has no kernel of its own for large launches: the
    ordinary one must be launched with its own units. Passes counting, applying, fused and single."""
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    from luminamoon_amd.optimizer import hip_backend
    from oracle import oracle as O

    group = group_dict(buffer=buffer, lr=1e-3, master_weights="full", **extra)
    cfg = oracle_config(O, group)
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    host = TensorSet(sizes, "f32", "f32", "f32", buffer in (2, "T2"), True, 81)
    dev, fill = _large(host)
    stepper = hip_backend.HipStepper()
    print(f"[case] f32 with master {buffer} {extra} tensors={count}", flush=True)
    for step in (1, 2, 3):
        grads = host.grads(step, 81)
        host.oracle_step(O, cfg, grads, step, threads=4)
        dev.hip_step(stepper, group, [g.cuda() for g in grads] + [fill], step)
        torch.cuda.synchronize()
        host.assert_equal(dev, f"step {step}")
    assert all(int(torch.count_nonzero(ws)) == 0 for ws in stepper.workspace._bufs.values())


# Waves whose elements leave optimistic lanes' ranges: the kernels compute them again on the general path.
def _exact_cancellation(host, grads):
    for m, g in zip(host.m, grads):  # m' or the direction near or at zero beside ordinary elements
        m[::97] = (g[::97].float() * -(1.0 - 0.81) / 0.81).to(m.dtype)


def _dead(host, grads):
    for i, g in enumerate(grads):  # zero gradients, m and v decayed to subnormals or zero
        g[::3] = 0.0
        host.m[i][::3] = 1e-44
        host.m[i][::6] = 0.0
        if host.v[i] is not None:
            host.v[i][::3] = 1e-41
            host.v[i][::9] = 0.0


def _specials(host, grads):
    for i, g in enumerate(grads):
        pos = [k for k in (3, 700, 1029, 2050, 3000, 4097) if k < g.numel()]
        _inject(g, pos, GRAD_SPECIALS, i)
        _inject(host.m[i], [p + 1 for p in pos if p + 1 < g.numel()], M_SPECIALS, i)
        _inject(host.p[i], [p + 2 for p in pos if p + 2 < g.numel()], P_SPECIALS, i)
        if host.v[i] is not None:
            _inject(host.v[i], [p + 3 for p in pos if p + 3 < g.numel()], V_SPECIALS, i)


def _scales(host, grads):
    for i, s in enumerate(host.sc):
        s[3] = [0.0, float("nan"), float("inf"), -1.3, 1e30, 1.3][i % 6]
    grads[1].zero_()


@pytest.mark.parametrize("inputs", [_exact_cancellation, _dead, _specials, _scales], ids=lambda f: f.__name__[1:])
@pytest.mark.parametrize("buffer,pdt,sdt", [
    (2, "bf16", "bf16"), (2, "bf16", "f32"), (2, "f16", "f32"), (1, "bf16", "bf16"), (1, "bf16", "f32"), (1, "f16", "f32"),
])
def test_optimistic_lanes_match_oracle(buffer, pdt, sdt, inputs):
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    from luminamoon_amd.optimizer import hip_backend
    from oracle import oracle as O

    for extra in ({}, {"bound_ratio": 1e-7}, {"eps": 1e-13}, {"betas": (0.0, 0.999)}, {"lr": 0.0}, {"lr": 1e-9}):
        group = group_dict(buffer=buffer, state_precision="param" if sdt != "f32" else "fp32", **{"lr": 1e-3, **extra})
        cfg = oracle_config(O, group)
        host = TensorSet([4096 + 37, 2048, 1000, 6144, 70_001, 512], pdt, pdt, sdt, buffer == 2, False, 79, m_scale=3e-4)
        for v in host.v:
            if v is not None:
                v.copy_((v.float() ** 2).to(v.dtype))
        # one step for fp16: a NaN's sign, which IEEE 754 leaves open, becomes the sign of a 65504
        steps = (2,) if pdt == "f16" else (2, 3)
        grads = [host.grads(s, 79) for s in steps]
        inputs(host, grads[0])
        dev, fill = _large(host)
        stepper = hip_backend.HipStepper()
        print(f"[case] lanes {buffer} {pdt}/{sdt} {inputs.__name__} {extra}", flush=True)
        for step, g in zip(steps, grads):
            host.oracle_step(O, cfg, g, step, threads=4)
            dev.hip_step(stepper, group, [x.cuda() for x in g] + [fill], step)
            torch.cuda.synchronize()
            for i in range(len(host.sizes)):
                for name in ("p", "m", "v", "sc"):
                    a, b = getattr(host, name)[i], getattr(dev, name)[i]
                    if a is not None:
                        _assert_same(a, b, f"{extra} step {step} {name}[{i}]")


# One of every large form: f32 state with and without a master, lanes with f32 and with 16-bit state.
FORMS = [
    (1, "f32", "f32", {}), (2, "f32", "f32", {}), ("T1", "f32", "f32", {}), ("T2", "f32", "f32", {}),
    ("T2", "bf16", "f32", {}), ("T2", "f16", "f32", {}),
    (2, "bf16", "f32", {"master_weights": "full"}), ("T2", "f16", "f32", {"master_weights": "semi"}),
    ("T1", "bf16", "f32", {"master_weights": "full"}), (1, "f16", "f32", {"master_weights": "full"}),
    (2, "bf16", "f32", {}), (2, "f16", "f32", {}), (1, "bf16", "f32", {}), (1, "f16", "f32", {}),
    (2, "bf16", "bf16", {"state_precision": "param"}), (1, "bf16", "bf16", {"state_precision": "param"}),
]
FORM_IDS = ["-".join(map(str, f[:3])) + ("-master" if "master_weights" in f[3] else "") for f in FORMS]


class _Case:
    """A form's tensors on the host and on the device, the device's as views at `offs` elements into their
    buffers and with one zero tensor of LARGE elements behind them; steps both and compares."""

    def __init__(self, form, sizes, offs=None, ranges=None, bases=None, **kw):
        from luminamoon_amd.optimizer import hip_backend
        from oracle import oracle as O

        buffer, pdt, sdt, extra = form
        self.O, n = O, len(sizes)
        self.group = group_dict(buffer=buffer, lr=1e-3, **{**extra, **kw})
        self.cfg = oracle_config(O, self.group)
        master = self.group["master_weights"] > 0
        self.host = TensorSet(sizes, pdt, pdt, sdt, buffer in (2, "T2"), master, 83, m_scale=3e-4)
        for v in self.host.v:
            if v is not None:
                v.copy_((v.float() ** 2).to(v.dtype))
        self.offs = offs or [0] * n
        self.ranges = ranges or [None] * n
        self.bases = bases or [0] * n
        self.dev, self.fill = _large(self.host)
        for xs in (self.dev.p, self.dev.m, self.dev.v, self.dev.mp):
            xs[:n] = [self._view(x, k) for x, k in zip(xs, self.offs)]
        self.tables = [torch.tensor(r, dtype=torch.int64, device="cuda") if r else None for r in self.ranges] + [None]
        self.stepper = hip_backend.HipStepper()

    @staticmethod
    def _view(x, k):
        if x is None:
            return None
        big = torch.zeros(x.numel() + 256, dtype=x.dtype, device="cuda")
        big[k:k + x.numel()] = x.to("cuda").reshape(-1)
        return big[k:k + x.numel()]

    def oracle(self, step):
        """One step on the host; inactive ranges are stepped with a zero gradient and put back."""
        h = self.host
        grads = h.grads(step, 84)
        kept = []
        for i, rs in enumerate(self.ranges):
            for b, e in rs or []:
                grads[i][b:e] = 0
                kept += [(xs[i], b, e, xs[i][b:e].clone()) for xs in (h.p, h.m, h.v, h.mp) if xs[i] is not None]
        self.O.step(self.cfg, h.p, grads, h.m, h.v, h.mp, h.sc, [step] * len(h.sizes), list(range(len(h.sizes))), threads=4,
                    index_bases=self.bases)
        for x, b, e, old in kept:
            x[b:e] = old
        return grads

    def device_grads(self, grads):
        return [self._view(g, k) for g, k in zip(grads, self.offs)] + [self.fill]

    def prepare(self, grads, step):
        d, n = self.dev, len(self.dev.sizes)
        return self.stepper.prepare(d.p, grads, d.m, d.v, d.mp, d.sc, [step] * n, list(range(n)), self.bases + [0], self.tables)

    def steps(self, steps, label):
        for step in steps:
            grads = self.device_grads(self.oracle(step))  # held until the step has run
            self.stepper.launch(self.group, self.prepare(grads, step))
            self.check(f"{label} step {step}")

    def check(self, label):
        torch.cuda.synchronize()
        self.host.assert_equal(self.dev, label)
        assert int(torch.count_nonzero(self.dev.m[-1])) == 0, label  # the zero tensor stayed zero
        assert all(int(torch.count_nonzero(ws)) == 0 for ws in self.stepper.workspace._bufs.values()), label


def _skip_without_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("form", FORMS, ids=FORM_IDS)
def test_large_views_inactive_ranges_and_index_bases(form, count):
    """Heads of 0 to 255 elements (views at +0 to +193, shorter tensors among them), inactive ranges over
    heads, part and whole units and the tensor's end, shards whose offsets pass 2^31; the first step counts
    and applies, the second is fused, the third keeps two passes."""
    _skip_without_gpu()
    sizes = [EDGES[i % len(EDGES)] for i in range(count)]
    offs = [(0, 1, 33, 63, 64, 130, 193)[i % 7] for i in range(count)]

    def ranges(i, n):
        if i % 3 == 0:
            return None
        if i % 11 == 1:
            return [(0, n)]
        rs = [(0, 2), (100, 190), (255, 1300), (2048, 5120), (6000, 6001), (n - 300, n)]
        out = []
        for b, e in rs:
            b, e = max(b, out[-1][1] + 1 if out else 0), min(e, n)
            if b < e:
                out.append((b, e))
        return out

    case = _Case(form, sizes, offs, [ranges(i, n) for i, n in enumerate(sizes)], [i * 0x13579BDF for i in range(count)])
    print(f"[case] views and ranges {form} tensors={count}", flush=True)
    case.steps((1, 2), f"{form}")
    case = _Case(form, sizes, offs, case.ranges, case.bases, fused_single_pass=False)
    case.steps((2,), f"{form} two passes")


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("form", FORMS, ids=FORM_IDS)
def test_large_single_pass_matches_oracle(form, count):
    """cautious=False: one pass that counts nothing, with views."""
    _skip_without_gpu()
    case = _Case(form, [EDGES[i % len(EDGES)] for i in range(count)], [(0, 1, 130)[i % 3] for i in range(count)], cautious=False)
    print(f"[case] single pass {form} tensors={count}", flush=True)
    case.steps((1, 2), f"{form}")


@pytest.mark.parametrize("count", [len(EDGES), 60], ids=["inline", "table"])
@pytest.mark.parametrize("form", [FORMS[1], FORMS[4], FORMS[6], FORMS[10], FORMS[14]], ids=lambda f: f"{f[0]}-{f[1]}-{f[2]}")
def test_large_launches_in_pieces_match_oracle(form, count, monkeypatch):
    """A unit space cut into launches of 6,001 blocks: tensors straddle the cuts."""
    _skip_without_gpu()
    monkeypatch.setenv("LV_MAX_GRID_BLOCKS", "6001")
    case = _Case(form, [EDGES[i % len(EDGES)] for i in range(count)], [(0, 1, 130)[i % 3] for i in range(count)])
    print(f"[case] pieces {form} tensors={count}", flush=True)
    case.steps((1, 2), f"{form}")


@pytest.mark.parametrize("form", FORMS, ids=FORM_IDS)
def test_large_graph_steps_match_oracle(form):
    """Steps from a device record, eagerly and as replays of a captured graph, with eager work between."""
    _skip_without_gpu()
    case = _Case(form, EDGES, [(0, 1, 130)[i % 3] for i in range(len(EDGES))])
    print(f"[case] graph {form}", flush=True)
    grads = case.oracle(2)
    static = case.device_grads(grads)
    prep = case.prepare(static, 0)
    rec = torch.zeros(4, dtype=torch.int64, device="cuda")
    rec[0] = 1
    ws = case.stepper.graph_workspace(case.group, prep)
    case.stepper.launch_graph(case.group, prep, rec, ws)
    case.check(f"{form} step 2")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        case.stepper.launch_graph(case.group, prep, rec, ws)
    for step in (3, 4, 5):
        for s, g in zip(static, case.oracle(step)):
            s.copy_(g)
        torch.cuda.synchronize()
        graph.replay()
        case.check(f"{form} replay of step {step}")
        assert int(rec[0]) == step and int(torch.count_nonzero(ws)) == 0
