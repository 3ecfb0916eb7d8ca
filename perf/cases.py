"""The optimizer steps this package is measured on: one steady `LuminaV.step()` per pass.

A case is a model's parameter list (the README's two tensors, ragged lists, GPT-2- and Llama-shaped
models), its dtypes and the optimizer's options. `prepare` builds the optimizer over it, takes the
first step (which sets up the state, the descriptors and the workspace, as in any training run) and
then fills every buffer with the values of a run under way, from the seed alone; `run` is one later
step. The step updates the params and the optimizer state in place, and those buffers are the outputs.

Unfused lists live in arenas, every tensor on a 256-element boundary of its own (torch's allocator
also starts each tensor on a 512-byte boundary); a fused list lives in LuminaV's own bucket. Either
way each kind of buffer is one flat tensor, so that a model of any number of tensors has few outputs.
"""
import math
import random
import warnings

import torch

from luminamoon_amd import LuminaV

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
PAD = 256          # elements between the starts of an unfused list's tensors are a multiple of this
CHUNK = 1 << 26    # elements made or checked at once
LR, BETAS, EPS, TAU, LAM, RATIO, CLAMP_MIN = 8e-4, (0.9, 0.999), 1e-8, 0.8, 0.3, 0.05, 0.5
LAGGED_CS, LAGGED_BS = 1.3, 0.9  # the previous step's cautious and radial scales

DEFAULTS = dict(buffer="2", pdt="f32", state="fp32", fused=False, master="none", bound="coordinate", cautious=True,
                sr=True, wd=0.08, two_pass=False, grad="normal")


def _case(name, **kw):
    c = dict(DEFAULTS, **kw)
    return dict(name=name, **c) if name else c


def listed():
    gpt2 = dict(shape="gpt2", layers=12, d=768, vocab=50257)
    llama1b = dict(shape="llama", layers=16, d=2048, ffn=5632, vocab=32000)
    return [
        # The README's example: a 650-parameter classifier. Launch and host latency are all there is.
        _case("readme_f32", shape="mlp", rows=64, cols=10),
        # Many small tensors of any size (a vision model's or an adapter's list), stepped unfused.
        _case("ragged64_tdclm_f32", shape="ragged", tensors=64, total=3_500_000, shape_seed=2, buffer="1", grad="zeros5"),
        # GPT-2 small trained in fp32 with the constructor's defaults: CLM, every tensor on its own.
        _case("gpt2_clm_f32", **gpt2),
        # The same model with bucket fusion.
        _case("gpt2_clm_f32_bucket", fused=True, **gpt2),
        # The radial bound (the norms of every tensor enter the step) on the same model.
        _case("gpt2_t2_f32_radial", buffer="T2", bound="radial", **gpt2),
        # A 1B Llama in bf16 with the constructor's defaults: CLM, fp32 state, unfused.
        _case("llama1b_clm_bf16", pdt="bf16", **llama1b),
        # The same with the reference's own state dtype (bf16 m and v).
        _case("llama1b_clm_bf16_state16", pdt="bf16", state="param", **llama1b),
        # T1 over one bf16 bucket: the lightest two-stream step per parameter.
        _case("llama1b_t1_bf16_bucket", pdt="bf16", buffer="T1", fused=True, **llama1b),
        # T2 with bf16 state over one bucket: the least memory a two-buffer step can take.
        _case("llama1b_t2_bf16_state16", pdt="bf16", buffer="T2", state="param", fused=True, **llama1b),
        # fp16 mixed precision: full fp32 master weights, fp32 state, unfused.
        _case("llama1b_t2_f16_master", pdt="f16", buffer="T2", master="full", **llama1b),
        # The exact (not lagged) cautious scale: counting pass and applying pass in every step.
        _case("llama1b_td_bf16_two_pass", pdt="bf16", buffer="1", two_pass=True, **llama1b),
        # Half of a 7B Llama, the largest: one bf16 bucket with fp32 state and heavy-tailed grads.
        _case("llama7b_half_t2_bf16", shape="llama", layers=16, d=4096, ffn=11008, vocab=32000, buffer="T2", pdt="bf16",
              fused=True, grad="t3"),
    ]


def draw(rng):
    """One more case: model sizes spread over their logarithm from a few hundred to 10^9 parameters,
    odd sizes among them, and the options that are used in earnest, defaults most often."""
    while True:
        total = int(2 ** rng.uniform(9.0, 30.0))
        kind = rng.choice(("ragged", "ragged", "gpt2", "llama"))
        if kind == "ragged":
            c = dict(shape="ragged", tensors=min(int(2 ** rng.uniform(0.0, 9.0)), max(1, total // 8)), total=total,
                     shape_seed=rng.randrange(1 << 20))
        else:
            layers = rng.randint(2, 24)
            # d from the total: about 12 d^2 per layer; odd multiples of 2 or 8 among them
            d = max(16, int(math.sqrt(total / (12.0 * layers))))
            d -= d % rng.choice((1, 2, 8, 64)) if d >= 64 else 0
            c = dict(shape=kind, layers=layers, d=d, vocab=rng.randint(97, max(98, 8 * d)))
            if kind == "llama":
                c["ffn"] = int(d * rng.uniform(2.0, 3.5))
        pdt = rng.choice(("f32", "bf16", "bf16", "f16"))
        c.update(buffer=rng.choice(("2", "2", "1", "T1", "T2", "T2")), pdt=pdt, fused=rng.random() < 0.4,
                 state="param" if rng.random() < 0.3 else "fp32",
                 master=rng.choice(("semi", "full")) if pdt != "f32" and rng.random() < 0.25 else "none",
                 bound=rng.choice(("radial", "none")) if rng.random() < 0.2 else "coordinate",
                 cautious=rng.random() < 0.85, sr=rng.random() < 0.9, wd=0.08 if rng.random() < 0.85 else 0.0,
                 two_pass=rng.random() < 0.15, grad=rng.choice(("normal", "normal", "zeros5", "t3")))
        c = _case("", **c)
        if 256 <= sum(map(math.prod, _shapes(c))) <= 1 << 30:
            return c


def _shapes(case):
    """The parameter shapes of a case's model."""
    kind = case["shape"]
    if kind == "mlp":
        return [(case["rows"], case["cols"]), (case["cols"],)]
    if kind == "ragged":  # log-uniform weights, scaled to the total
        r = random.Random(case["shape_seed"])
        w = [math.exp(r.uniform(0.0, math.log(2.0 ** 14))) for _ in range(case["tensors"])]
        return [(max(1, int(case["total"] * x / sum(w))),) for x in w]
    d, v = case["d"], case["vocab"]
    if kind == "gpt2":
        block = [(d,), (d, 3 * d), (d, d), (d,), (d, 4 * d), (4 * d, d)]
        return [(v, d)] + block * case["layers"] + [(d,)]
    f = case["ffn"]
    block = [(d, d)] * 4 + [(f, d), (f, d), (d, f), (d,), (d,)]
    return [(v, d)] + block * case["layers"] + [(d,), (v, d)]


def _spans(case):
    """[begin, end) of every tensor in the case's flat buffers, and the buffers' length."""
    spans, off = [], 0
    for n in map(math.prod, _shapes(case)):
        spans.append((off, off + n))
        off += n if case["fused"] else -(-n // PAD) * PAD
    return spans, off


def _dual(case):
    return case["buffer"] in ("2", "T2")


def _masters(case):
    return case["master"] != "none" and case["pdt"] != "f32"


def _state_is_16bit(case):
    return case["pdt"] != "f32" and case["state"] == "param" and case["master"] != "full"


def _fill(case, seed, bufs):
    """Fills the flat buffers with a run's values: params around 0.02, grads around 1e-3 (normal, 5%
    exact zeros, or heavy-tailed), the first moment of such grads, and their second moment."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n = bufs["p"].numel()
    for a in range(0, n, CHUNK):
        b = min(n, a + CHUNK)

        def noise():
            return torch.randn(b - a, generator=gen, device="cuda")

        p = noise().mul_(0.02)
        bufs["p"][a:b] = p
        if "mp" in bufs:
            bufs["mp"][a:b] = p
        g = noise()
        if case["grad"] == "zeros5":
            g.masked_fill_(torch.rand(b - a, generator=gen, device="cuda") < 0.05, 0.0)
        elif case["grad"] == "t3":
            g.div_((noise().square_().add_(noise().square_()).add_(noise().square_())).div_(3.0).sqrt_())
        bufs["g"][a:b] = g.mul_(1e-3)
        bufs["m"][a:b] = noise().mul_(3e-4)
        if "v" in bufs:
            bufs["v"][a:b] = torch.rand(b - a, generator=gen, device="cuda").add_(0.5).mul_(1e-6)
    bufs["scratch"].zero_()
    bufs["scratch"][:, 3] = LAGGED_CS if case["cautious"] else 1.0
    bufs["scratch"][:, 4] = LAGGED_BS if case["bound"] == "radial" else 1.0


def _empty(case, n, rows):
    """Flat buffers of n elements, zeroed."""
    pdt = DTYPES[case["pdt"]]
    sdt = torch.bfloat16 if _state_is_16bit(case) else torch.float32  # an fp16 container holds bf16 bits
    bufs = {"p": torch.zeros(n, dtype=pdt, device="cuda"), "g": torch.zeros(n, dtype=pdt, device="cuda"),
            "m": torch.zeros(n, dtype=sdt, device="cuda")}
    if _dual(case):
        bufs["v"] = torch.zeros(n, dtype=sdt, device="cuda")
    if _masters(case):
        bufs["mp"] = torch.zeros(n, dtype=torch.float32, device="cuda")
    bufs["scratch"] = torch.zeros(rows, 128, dtype=torch.float32, device="cuda")
    return bufs


def _optimizer(case, params, total):
    buffer = int(case["buffer"]) if case["buffer"] in ("1", "2") else case["buffer"]
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")  # the fusion advice
        return LuminaV(params, lr=LR, betas=BETAS, eps=EPS, weight_decay=case["wd"], tau=TAU, lam=LAM, buffer=buffer,
                       cautious=case["cautious"], cautious_clamp_min=CLAMP_MIN, stochastic_rounding=case["sr"],
                       bound=case["bound"] != "none", bound_type="radial" if case["bound"] == "radial" else "coordinate",
                       bound_ratio=RATIO, master_weights=case["master"], fused_single_pass=not case["two_pass"],
                       state_precision=case["state"], fuse_tensors=case["fused"],
                       bucket_cap_mb=max(500.0, 4.0 * total / (1 << 20) + 1.0))


def prepare(case, seed):
    spans, total = _spans(case)
    shapes = _shapes(case)
    sdt = torch.float16 if case["pdt"] == "f16" else torch.bfloat16  # 16-bit state is in the param dtype
    if case["fused"]:
        pdt = DTYPES[case["pdt"]]
        params = [torch.nn.Parameter(torch.full(s, 0.02, dtype=pdt, device="cuda")) for s in shapes]
        for p in params:
            p.grad = torch.full_like(p, 1e-3)
        opt = _optimizer(case, params, total)

        def flat(t):  # a bucket's tensors are views of one flat buffer
            return t.detach().as_strided((total,), (1,), 0)

        st = opt.state[params[0]]
        bufs = {"p": flat(params[0]), "g": flat(params[0].grad), "m": flat(st["exp_avg"])}
        if _dual(case):
            bufs["v"] = flat(st["exp_avg_sq"])
        if _masters(case):
            bufs["mp"] = flat(st["master_param"])
        bufs["scratch"] = st["scratch"].view(1, 6)
    else:
        bufs = _empty(case, total, len(shapes))
        bufs["p"].fill_(0.02)
        bufs["g"].fill_(1e-3)

        def part(name, k):
            a, b = spans[k]
            t = bufs[name][a:b].view(shapes[k])
            return t.view(sdt) if name in "mv" and _state_is_16bit(case) else t

        params = [torch.nn.Parameter(part("p", k)) for k in range(len(shapes))]
        for k, p in enumerate(params):
            p.grad = part("g", k)
        opt = _optimizer(case, params, total)
        for k, p in enumerate(params):
            st = {"step": 0, "scratch": bufs["scratch"][k, :6], "exp_avg": part("m", k),
                  "buf_count": opt.param_groups[0]["buffer"]}
            if _dual(case):
                st["exp_avg_sq"] = part("v", k)
            if _masters(case):
                st["master_param"] = part("mp", k)
                part("mp", k).copy_(p.detach())
            st["scratch"].copy_(torch.tensor([0.0, 0.0, 0.0, 1.0, 1.0, 0.0]))
            opt.state[p] = st
    opt.step()  # the first step of the run: state, descriptors, workspace
    views = {k: (b.view(torch.bfloat16) if k in "mv" and b.dtype == torch.float16 else b) for k, b in bufs.items()}
    _fill(case, seed, views)
    return {"opt": opt, "params": params, "out": {k: b for k, b in views.items() if k != "g"}}


def run(state):
    state["opt"].step()
    return state["out"]


def work(case):
    n = sum(map(math.prod, _shapes(case)))
    pb = 4 if case["pdt"] == "f32" else 2
    sb = 2 if _state_is_16bit(case) else 4
    states = 2 if _dual(case) else 1
    # grad read, param written and read (or, with a master, the master read and written), state both
    per = pb + pb + (8 if _masters(case) else pb) + 2 * sb * states
    ops = {"2": 75, "1": 50, "T1": 30, "T2": 40}[case["buffer"]] + (15 if pb == 2 and case["sr"] else 0)
    return {"bytes": float(n * per), "flops": float(n * ops)}


def tolerance(case):
    """f32 buffers: the rounding of some forty f32 operations (at most 3.6e-8 off `exact`, measured).
    16-bit buffers: a value whose f32 result moves by a rounding may take the other 16-bit neighbour
    (against `exact`, whose values are not rounded to 16 bits at all: 2.3e-3 for bf16 and 2e-4 for fp16
    params, measured); the largest difference is one or two units in the last place."""
    if case["pdt"] == "f32":
        return {"rel": 2e-7, "max": 1e-5}
    if case["pdt"] == "f16" and not _state_is_16bit(case):
        return {"rel": 1e-3, "max": 4e-3}
    return {"rel": 1e-2, "max": 2e-2}


# ---------------------------------------------------------------------------- the step in 64 bits


def _f32(x):
    return float(torch.tensor(x, dtype=torch.float32))


def _tanh_pade(x):
    """The algorithm's tanh: a [13/6] Pade form with f32 coefficients."""
    x = x.clamp(-_f32(7.9988117), _f32(7.9988117))
    x2 = x * x
    p = torch.full_like(x, _f32(-2.7607684e-16))
    for c in (2.000188e-13, -8.604672e-11, 5.122297e-8, 1.4857224e-5, 6.3726193e-4, 4.8935246e-3):
        p = p * x2 + _f32(c)
    q = torch.full_like(x, _f32(1.1982584e-6))
    for c in (1.1853471e-4, 2.2684346e-3, 4.8935246e-3):
        q = q * x2 + _f32(c)
    return x * p / q


def _direction(case, g, m, v):
    """u, m', v' of the second step for f64 values."""
    b1, b2, eps, tau, lam = _f32(BETAS[0]), _f32(BETAS[1]), _f32(EPS), _f32(TAU), _f32(LAM)
    bc1, bc2 = 1.0 - b1 ** 3, 1.0 - b2 ** 2
    clamp_v = case["pdt"] == "f16"
    m2 = b1 * m + (1.0 - b1) * g
    if case["buffer"] == "2":
        clm = b1 * m2 + (1.0 - b1) * g
        v2 = b2 * v + (1.0 - b2) * (g - m2).square()
        v2 = v2.clamp(max=65000.0) if clamp_v else v2
        sigma = v2.clamp(min=0.0).sqrt() * (bc1 * tau / math.sqrt(bc2)) + eps * bc1 * tau
        return _tanh_pade(clm / sigma.clamp(min=1e-12)), m2, v2
    clm = b1 * b1 * m + (1.0 - b1 * b1) * g
    env = b1 * b1 * m.abs() + (1.0 - b1 * b1) * g.abs() + eps
    if case["buffer"] == "T2":
        v2 = b2 * v + (1.0 - b2) * (g - m).square()
        v2 = v2.clamp(max=65000.0) if clamp_v else v2
        env = env + 0.5 * lam * (g - m).abs() + 0.5 * lam / math.sqrt(bc2) * v2.clamp(min=0.0).sqrt()
        return clm / env, m2, v2
    return clm / (env + lam * (g - m).abs()), m2, None


def _bounded(case, step, p):
    """The coordinate bound and, for fp16 params, the fp16 safety bound of a step."""
    tri = case["buffer"] in ("T1", "T2")

    def bound(step, b):
        if tri:
            bb = b * (b + step.abs())
            return bb * step / (step * step + bb)
        return b * _tanh_pade(step / b)

    if case["bound"] == "coordinate":
        step = bound(step, _f32(RATIO) * ((p.abs() + _f32(1e-2)) if tri else (p * p + _f32(1e-4)).sqrt()))
    if case["pdt"] == "f16":
        step = bound(step, (p.abs() * _f32(0.01)).clamp(min=_f32(1.5e-4)))
    return step


def _radial(case, u_sq, p_sq, cs):
    radius = RATIO * max(math.sqrt(p_sq), 1.0)
    r = LR * math.sqrt(u_sq) * cs / radius
    if case["buffer"] in ("T1", "T2"):
        return (1.0 + r) / (r * r + 1.0 + r)
    return 1.0 if r < 1e-4 else float(_tanh_pade(torch.tensor(r, dtype=torch.float64))) / r


def exact(case, seed):
    spans, total = _spans(case)
    if total > 1 << 30:
        return None  # the f64 copies of the largest model would not fit beside everything else
    bufs = _empty(case, total, 1 if case["fused"] else len(spans))
    if case["fused"]:
        bufs["scratch"] = bufs["scratch"][:, :6].contiguous()
        spans = [(0, total)]
    _fill(case, seed, bufs)
    out = {k: b.double() for k, b in bufs.items() if k != "g"}
    lr, wd = _f32(LR), _f32(case["wd"])
    cautious, radial = case["cautious"], case["bound"] == "radial"
    ema = 0.95 if case["buffer"] in ("1", "T1") else 0.80
    old_p = bufs["mp"] if _masters(case) else bufs["p"]
    for k, (begin, end) in enumerate(spans):
        chunks = [(a, min(end, a + CHUNK)) for a in range(begin, end, CHUNK)]

        def values(a, b):
            g, m = bufs["g"][a:b].double(), bufs["m"][a:b].double()
            u, m2, v2 = _direction(case, g, m, bufs["v"][a:b].double() if _dual(case) else None)
            mask = u * g > 0.0
            return (u * mask if cautious else u), m2, v2, mask

        count, u_sq, p_sq = 0, 0.0, 0.0
        if cautious or radial:
            for a, b in chunks:
                u, _, _, mask = values(a, b)
                count += int(mask.sum())
                if radial:
                    u_sq += float(u.square().sum())
                    p_sq += float(old_p[a:b].double().square().sum())
        scale = 1.0 / min(max(count / (end - begin), CLAMP_MIN), 1.0)
        s = out["scratch"][k]
        if case["two_pass"]:
            cs = scale if cautious else 1.0
            bs = _radial(case, u_sq, p_sq, cs) if radial else 1.0
            new = (cs, bs)
        else:
            cs, bs = float(s[3]), float(s[4])
            c2 = ema * cs + (1.0 - ema) * scale if cautious else 1.0
            new = (c2, ema * bs + (1.0 - ema) * _radial(case, u_sq, p_sq, c2) if radial else 1.0)
        for a, b in chunks:
            u, m2, v2, _ = values(a, b)
            p = old_p[a:b].double()
            step = lr * u * (cs if cautious else 1.0)
            step = _bounded(case, step * bs if radial else step, p)
            p = p - lr * wd * p - step
            out["p"][a:b] = p
            if _masters(case):
                out["mp"][a:b] = p
            out["m"][a:b] = m2
            if _dual(case):
                out["v"][a:b] = v2
        s[3], s[4] = new
    return out
