"""The decoder's workloads, as the performance of this package is measured on them.

Whole calls: serving one short and one ordinary utterance, the training step of
the benchmark (8 utterances of 512 frames, every grad on) and one DecoderLora
step over the frozen decoder. Layers, each through the C ABI entry point that a
program calls: the generator's resblock convs with the AdaIN fused into them
(forward and backward), a backbone conv, an upsampler, AdaIN + Snake, the
spectral head and the style projection. Sizes follow the decoder's own: stage 0
has 256 channels and 20 T positions, stage 1 has 128 channels and 120 T + 1, the
backbone T or 2 T positions.
"""
import ctypes
import math

import torch
import torch.nn.functional as F

from brosoundml_amd import config, native

CFG = config.KOKORO
P = native.ptr
EPS = 1e-5


def listed():
    return [
        # serving a word or two: the shortest calls, where launches and latency count
        {"name": "infer_b1_t21", "kind": "infer", "n": 1, "t": 21},
        # serving a sentence of five seconds
        {"name": "infer_b1_t200", "kind": "infer", "n": 1, "t": 200},
        # the training step of the benchmark: the largest call
        {"name": "train_b8_t512", "kind": "train", "n": 8, "t": 512},
        # fine-tuning the style adapters on two short utterances
        {"name": "lora_b2_t64", "kind": "lora", "n": 2, "t": 64},
        # the widest resblock conv of stage 1 on the training batch, feeding an AdaIN
        {"name": "resconv_fwd_s1_k11", "kind": "resconv_fwd", "n": 8, "c": 128, "l": 61441, "k": 11, "d": 5, "res": False},
        # stage 0's narrowest for one utterance of four seconds, with the block's skip
        {"name": "resconv_fwd_s0_k3", "kind": "resconv_fwd", "n": 1, "c": 256, "l": 3220, "k": 3, "d": 1, "res": True},
        # the backward of such a unit, odd rows: input grad with the AdaIN + Snake backward, and weight grad
        {"name": "resconv_bwd_s1_k7", "kind": "resconv_bwd", "n": 2, "c": 128, "l": 24121, "k": 7, "d": 3},
        # a decode block's first conv (1024 + 64 + 2 input channels) on ragged short rows, forward and backward
        {"name": "backbone_b4_l331", "kind": "conv", "n": 4, "ci": 1090, "co": 1024, "l": 331, "k": 3},
        # the first upsampler, forward and backward
        {"name": "ups0_b4_l512", "kind": "convt", "n": 4, "ci": 512, "co": 256, "l": 512, "k": 20, "s": 10},
        # AdaIN + Snake on two seconds at 24 kHz, forward and backward
        {"name": "adain_snake_l48000", "kind": "adain", "n": 1, "c": 256, "l": 48000},
        # the spectral head of the training batch, forward and backward
        {"name": "spectral_b8_l61441", "kind": "spectral", "n": 8, "l": 61441},
        # every AdaIN unit's style projection at once, forward and backward
        {"name": "style_b8", "kind": "style", "n": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["infer", "infer", "train", "lora", "resconv_fwd", "resconv_fwd", "resconv_bwd", "resconv_bwd",
                       "conv", "convt", "adain", "spectral", "style"])
    n = rng.randint(1, 8)
    if kind == "infer":
        return {"kind": kind, "n": n, "t": _log(rng, 8, 512)}
    if kind == "train":
        return {"kind": kind, "n": n, "t": _log(rng, 16, 512)}
    if kind == "lora":
        n = rng.randint(1, 4)
        return {"kind": kind, "n": n, "t": _log(rng, 16, 256 // n)}
    if kind in ("resconv_fwd", "resconv_bwd"):
        t = _log(rng, 8, 512)
        stage = rng.randint(0, 1)
        c = {"kind": kind, "n": n, "c": 128 if stage else 256, "l": 120 * t + 1 if stage else 20 * t,
             "k": rng.choice([3, 7, 11]), "d": rng.choice([1, 3, 5])}
        if kind == "resconv_fwd":
            c["res"] = rng.random() < 0.5
        return c
    if kind == "conv":
        ci, co = rng.choice([(514, 1024), (1090, 1024), (1024, 1024), (1090, 512), (512, 512)])
        return {"kind": kind, "n": n, "ci": ci, "co": co, "l": _log(rng, 16, 1024), "k": 3}
    if kind == "convt":
        ci, co, k, s, up = rng.choice([(512, 256, 20, 10, 2), (256, 128, 12, 6, 20)])
        return {"kind": kind, "n": n, "ci": ci, "co": co, "l": up * _log(rng, 8, 512), "k": k, "s": s}
    if kind == "adain":
        return {"kind": kind, "n": n, "c": rng.choice([128, 256, 512]), "l": _log(rng, 300, 61441)}
    if kind == "spectral":
        return {"kind": kind, "n": n, "l": 120 * _log(rng, 8, 512) + 1}
    return {"kind": kind, "n": n + 8 * rng.randint(0, 3)}


# ─── inputs ──────────────────────────────────────────────────────────────────


class _Gen:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda") * (hi - lo) + lo


class _Raw:
    def __init__(self, address, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (address, False), "version": 2}


def _view(owner, address, *shape):
    """The device floats at an address, as a tensor over the same memory; the tensor keeps their owner alive."""
    t = torch.as_tensor(_Raw(address, shape), device="cuda")
    t.owner = owner
    return t


def _param_views(model):
    return {name: _view(model, model.ctx.L.kdec_model_param_ptr(model.h, name.encode()), r, c)
            for name, (r, c) in model.param_shapes().items()}


def _model(g):
    """A decoder at the Kokoro sizes with random weights (PyTorch's default bounds; Snake alphas in [0.5, 2])."""
    ctx = native.Context(0)
    model = native.Model(ctx, CFG)
    shapes = model.param_shapes()
    for name, v in _param_views(model).items():
        if ".alpha" in name:
            v.uniform_(0.5, 2.0, generator=g.g)
            continue
        w = name[: -len(".bias")] + ".weight" if name.endswith(".bias") else name
        bound = 1.0 / math.sqrt(shapes[w][1] if w in shapes else shapes[name][1])
        v.uniform_(-bound, bound, generator=g.g)
    return ctx, model


def _utterances(g, n, t):
    f0 = g.uniform(80.0, 300.0, n, 2 * t)
    f0[g.uniform(0.0, 1.0, n, 2 * t) < 0.2] = 0.0  # unvoiced frames
    return {"asr": g.normal(n, CFG["asr_dim"], t), "f0": f0, "nn": g.normal(n, 2 * t, std=0.5),
            "style": g.normal(n, CFG["style_dim"], std=0.3)}


def prepare(case, seed):
    g = _Gen(seed)
    kind, n = case["kind"], case["n"]
    s = {"kind": kind, "case": case}
    if kind in ("infer", "train", "lora"):
        t = case["t"]
        s["ctx"], s["model"] = ctx, model = _model(g)
        s.update(_utterances(g, n, t))
        lens = config.lengths(CFG, t)
        s["audio"] = torch.empty(n, lens["audio"], device="cuda")
        if kind == "train":
            s["daudio"] = g.normal(n, lens["audio"])
            s["dstyle"] = torch.empty(n, CFG["style_dim"], device="cuda")
            first = model.param_shapes().__iter__().__next__()
            s["grads"] = _view(model, ctx.L.kdec_model_grad_ptr(model.h, first.encode()), ctx.L.kdec_model_param_total(model.h))
        if kind == "lora":
            s["daudio"] = g.normal(n, lens["audio"])
            s["har"] = g.normal(n, CFG["n_fft"] + 2, lens["frames"], std=0.3)
            s["cond"] = g.normal(n, 3)
            s["lora"] = lora = native.DecoderLora(model, 4, 0.5, seed=1)
            for name in ("A", "B", "W1", "W2"):
                p, r, c = lora.tensor(name)
                _view(lora, p, r, c).normal_(0.0, 0.3 if name[0] == "W" else 0.1, generator=g.g)
            s["out"] = {}
            for name in ("dA", "dB", "dW1", "dW2"):
                p, r, c = lora.tensor(name)
                s["out"][name] = _view(lora, p, r, c)
        torch.cuda.synchronize()
        return s
    s["ctx"] = native.Context(0)
    if kind == "resconv_fwd":
        c, l, k = case["c"], case["l"], case["k"]
        b = 1.0 / math.sqrt(c * k)
        s.update(x=g.normal(n, c, l), w=g.uniform(-b, b, c, c * k), b=g.uniform(-b, b, c),
                 r=g.normal(n, c, l) if case["res"] else None, y=torch.empty(n, c, l, device="cuda"),
                 stats=torch.empty(n * c, 2, device="cuda"))
    elif kind == "resconv_bwd":
        c, l, k = case["c"], case["l"], case["k"]
        b = 1.0 / math.sqrt(c * k)
        s.update(x=g.normal(n, c, l), dy=g.normal(n, c, l, std=0.1), w=g.uniform(-b, b, c, c * k),
                 gb=g.normal(n, 2 * c, std=0.3), alpha=g.uniform(0.5, 2.0, c), stats=torch.empty(n * c, 2, device="cuda"),
                 act=g.normal(n, c, l), r=g.normal(n, c, l, std=0.1))
        s["ctx"].call("kdec_instnorm_stats", P(s["x"]), c * l, n, c, l, EPS, P(s["stats"]))
        s.update(dx=torch.empty(n, c, l, device="cuda"), dgb=torch.empty(n, 2 * c, device="cuda"),
                 sums=torch.empty(c * c * k + 2 * c, device="cuda"))
    elif kind == "conv":
        ci, co, l, k = case["ci"], case["co"], case["l"], case["k"]
        b = 1.0 / math.sqrt(ci * k)
        s.update(x=g.normal(n, ci, l), w=g.uniform(-b, b, co, ci * k), b=g.uniform(-b, b, co), r=g.normal(n, co, l),
                 dy=g.normal(n, co, l, std=0.1), y=torch.empty(n, co, l, device="cuda"),
                 dx=torch.empty(n, ci, l, device="cuda"), sums=torch.empty(co * ci * k + co, device="cuda"))
    elif kind == "convt":
        ci, co, l, k, st = case["ci"], case["co"], case["l"], case["k"], case["s"]
        b = 1.0 / math.sqrt(co * k)
        s.update(x=g.normal(n, ci, l), w=g.uniform(-b, b, ci, co * k), b=g.uniform(-b, b, co),
                 dy=g.normal(n, co, l * st, std=0.1), y=torch.empty(n, co, l * st, device="cuda"),
                 dx=torch.empty(n, ci, l, device="cuda"), sums=torch.empty(ci * co * k + co, device="cuda"))
    elif kind == "adain":
        c, l = case["c"], case["l"]
        s.update(x=g.normal(n, c, l) * 1.5 + 0.3, dy=g.normal(n, c, l), gb=g.normal(n, 2 * c, std=0.3),
                 alpha=g.uniform(0.5, 2.0, c), stats=torch.empty(n * c, 2, device="cuda"),
                 y=torch.empty(n, c, l, device="cuda"), dx=torch.empty(n, c, l, device="cuda"),
                 dgb=torch.empty(n, 2 * c, device="cuda"), dalpha=torch.empty(c, device="cuda"))
    elif kind == "spectral":
        l, nf, hop = case["l"], CFG["n_fft"], CFG["hop"]
        s.update(post=g.normal(n, nf + 2, l, std=0.5), da=g.normal(n, (l - 1) * hop),
                 audio=torch.empty(n, (l - 1) * hop, device="cuda"), dpost=torch.empty(n, nf + 2, l, device="cuda"))
    else:
        r, sd = config.affine_rows(CFG), CFG["style_dim"]
        s.update(w=g.uniform(-0.09, 0.09, r, sd), b=g.uniform(-0.09, 0.09, r), style=g.normal(n, sd, std=0.3),
                 dgb=g.normal(n, r), gb=torch.empty(n, r, device="cuda"), dstyle=torch.empty(n, sd, device="cuda"),
                 sums=torch.empty(r * sd + r, device="cuda"))
    torch.cuda.synchronize()
    return s


def _at(t, off):
    return ctypes.c_void_p(t.data_ptr() + 4 * off)


def run(s):
    kind, case, call = s["kind"], s["case"], s["ctx"].call
    n = case["n"]
    if kind == "infer":
        m = s["model"]
        m.ctx.check(m.ctx.L.kdec_model_infer(m.h, n, case["t"], P(s["asr"]), P(s["f0"]), P(s["nn"]), P(s["style"]), None,
                                             P(s["audio"])))
        return s["audio"]
    if kind == "train":
        m = s["model"]
        m.zero_grad()
        m.forward(s["asr"], s["f0"], s["nn"], s["style"], case["t"], audio=s["audio"])
        m.backward(s["daudio"], wgrad=True, dalpha=True, dstyle=s["dstyle"])
        return {"audio": s["audio"], "dstyle": s["dstyle"], "grads": s["grads"]}
    if kind == "lora":
        d = s["lora"]
        d.zero_grad()
        d.forward(s["asr"], s["f0"], s["nn"], s["style"], case["t"], s["cond"], har=s["har"], audio=s["audio"])
        d.backward(s["daudio"])
        return {"audio": s["audio"], **s["out"]}
    if kind == "resconv_fwd":
        c, l, k, d = case["c"], case["l"], case["k"], case["d"]
        call("kdec_conv1d_fwd_stats", P(s["x"]), c * l, P(s["w"]), P(s["b"]), P(s["y"]), c * l, n, c, l, c, k, 1,
             d * (k - 1) // 2, d, P(s["r"]), c * l, 1.0, EPS, P(s["stats"]))
        return {"y": s["y"], "stats": s["stats"]}
    if kind == "resconv_bwd":
        c, l, k, d = case["c"], case["l"], case["k"], case["d"]
        nw, p = c * c * k, d * (k - 1) // 2
        call("kdec_fill", P(s["sums"]), nw + 2 * c, 0.0)
        call("kdec_conv1d_dgrad_adain_bwd", P(s["w"]), P(s["dy"]), c * l, n, c, l, c, k, 1, p, d, P(s["x"]), c * l,
             P(s["stats"]), P(s["gb"]), _at(s["gb"], c), 2 * c, 2, 0.0, P(s["alpha"]), P(s["r"]), c * l, P(s["dx"]), c * l,
             P(s["dgb"]), _at(s["dgb"], c), 2 * c, _at(s["sums"], nw + c))
        call("kdec_conv1d_wgrad", P(s["act"]), c * l, P(s["dy"]), c * l, P(s["sums"]), _at(s["sums"], nw), n, c, l, c, k, 1,
             p, d)
        return {"dx": s["dx"], "dgb": s["dgb"], "dw": s["sums"][:nw], "db": s["sums"][nw:nw + c],
                "dalpha": s["sums"][nw + c:]}
    if kind == "conv":
        ci, co, l, k = case["ci"], case["co"], case["l"], case["k"]
        nw = co * ci * k
        call("kdec_conv1d_fwd", P(s["x"]), ci * l, P(s["w"]), P(s["b"]), P(s["y"]), co * l, n, ci, l, co, k, 1, k // 2, 1,
             P(s["r"]), co * l, math.sqrt(0.5), 0.0)
        call("kdec_conv1d_dgrad", P(s["w"]), P(s["dy"]), co * l, P(s["dx"]), ci * l, n, ci, l, co, k, 1, k // 2, 1, 1.0, 0.0)
        call("kdec_fill", P(s["sums"]), nw + co, 0.0)
        call("kdec_conv1d_wgrad", P(s["x"]), ci * l, P(s["dy"]), co * l, P(s["sums"]), _at(s["sums"], nw), n, ci, l, co, k,
             1, k // 2, 1)
        return {"y": s["y"], "dx": s["dx"], "dw": s["sums"][:nw], "db": s["sums"][nw:]}
    if kind == "convt":
        ci, co, l, k, st = case["ci"], case["co"], case["l"], case["k"], case["s"]
        lo, nw, p = l * st, ci * co * k, (k - st) // 2
        call("kdec_convt1d_fwd", P(s["x"]), ci * l, P(s["w"]), P(s["b"]), P(s["y"]), co * lo, n, ci, l, co, k, st, p, 0)
        call("kdec_convt1d_dgrad", P(s["w"]), P(s["dy"]), co * lo, P(s["dx"]), ci * l, n, ci, l, co, k, st, p, 0)
        call("kdec_fill", P(s["sums"]), nw + co, 0.0)
        call("kdec_convt1d_wgrad", P(s["x"]), ci * l, P(s["dy"]), co * lo, P(s["sums"]), _at(s["sums"], nw), n, ci, l, co, k,
             st, p, 0)
        return {"y": s["y"], "dx": s["dx"], "dw": s["sums"][:nw], "db": s["sums"][nw:]}
    if kind == "adain":
        c, l = case["c"], case["l"]
        call("kdec_adain_act_fwd_stats", P(s["x"]), c * l, EPS, P(s["stats"]), P(s["gb"]), _at(s["gb"], c), 2 * c, 2, 0.0,
             P(s["alpha"]), P(s["y"]), c * l, None, 0, n, c, l)
        call("kdec_fill", P(s["dalpha"]), c, 0.0)
        call("kdec_adain_act_bwd", P(s["x"]), c * l, P(s["stats"]), P(s["gb"]), _at(s["gb"], c), 2 * c, 2, 0.0,
             P(s["alpha"]), P(s["dy"]), c * l, None, 0, P(s["dx"]), c * l, P(s["dgb"]), _at(s["dgb"], c), 2 * c,
             P(s["dalpha"]), n, c, l)
        return {k: s[k] for k in ("y", "stats", "dx", "dgb", "dalpha")}
    if kind == "spectral":
        l, nf, hop = case["l"], CFG["n_fft"], CFG["hop"]
        call("kdec_spectral_fwd", P(s["post"]), (nf + 2) * l, None, P(s["audio"]), (l - 1) * hop, n, l, nf, hop)
        call("kdec_spectral_bwd", P(s["post"]), (nf + 2) * l, None, P(s["da"]), (l - 1) * hop, P(s["dpost"]), (nf + 2) * l, n,
             l, nf, hop)
        return {"audio": s["audio"], "dpost": s["dpost"]}
    r, sd = s["w"].shape
    call("kdec_style_proj_fwd", P(s["w"]), P(s["b"]), P(s["style"]), sd, P(s["gb"]), r, n, r, sd)
    call("kdec_fill", P(s["sums"]), r * sd + r, 0.0)
    call("kdec_style_proj_bwd", P(s["w"]), P(s["style"]), sd, P(s["dgb"]), r, P(s["dstyle"]), sd, 0.0, P(s["sums"]),
         _at(s["sums"], r * sd), n, r, sd)
    return {"gb": s["gb"], "dstyle": s["dstyle"], "dw": s["sums"][:r * sd], "db": s["sums"][r * sd:]}


# ─── what a pass cannot do without ───────────────────────────────────────────


def _conv_macs(t):
    """Multiply-adds of the decoder's convs for one utterance of t frames."""
    c = CFG
    total = 2 * 3 * t + c["asr_dim"] * c["asr_res_dim"] * t  # F0 / N convs, asr_res
    cin, cout, l, cat = c["asr_dim"] + 2, c["enc_dim"], t, c["asr_res_dim"] + 2

    def block(ci, co, li, lo):
        return ci * co * 3 * lo + co * co * 3 * lo + (ci * co * lo if ci != co else 0)

    total += block(cin, cout, l, l)
    prev, res = cout, True
    for i in range(c["n_decode"]):
        up = i == c["dec_up_at"]
        lo = 2 * l if up else l
        total += block(prev + (cat if res else 0), c["dec_out"][i], l, lo)
        prev, l, res = c["dec_out"][i], lo, res and not up
    har = c["n_fft"] + 2
    for i in range(c["n_ups"]):
        u, ku, ch = c["ups_rates"][i], c["ups_kernels"][i], prev // 2
        total += prev * ch * ku * l
        l = l * u + (1 if i + 1 == c["n_ups"] else 0)
        rest = math.prod(c["ups_rates"][i + 1:c["n_ups"]])
        total += har * ch * (2 * rest if rest > 1 else 1) * l
        total += 6 * ch * ch * (7 if i + 1 < c["n_ups"] else 11) * l
        total += sum(6 * ch * ch * k * l for k in c["rb_kernels"][:c["n_kernels"]])
        prev = ch
    return total + prev * har * c["conv_post_k"] * l


def work(case):
    kind, n = case["kind"], case["n"]
    if kind in ("infer", "train", "lora"):
        t = case["t"]
        params = 53251204
        io = n * (CFG["asr_dim"] * t + 4 * t + CFG["style_dim"] + config.lengths(CFG, t)["audio"])
        flops = 2.0 * n * _conv_macs(t)
        if kind == "infer":
            return {"bytes": 4.0 * (params + io), "flops": flops}
        if kind == "train":  # forward, input grads, weight grads
            return {"bytes": 4.0 * (2 * params + 2 * io), "flops": 3 * flops}
        return {"bytes": 4.0 * (params + 2 * io), "flops": 2 * flops}
    if kind == "resconv_fwd":
        c, l, k = case["c"], case["l"], case["k"]
        return {"bytes": 4.0 * (n * c * l * (3 if case["res"] else 2) + c * c * k), "flops": 2.0 * n * c * c * k * l}
    if kind == "resconv_bwd":  # dy, x, the conv's input and the skip's grad in, dx out
        c, l, k = case["c"], case["l"], case["k"]
        return {"bytes": 4.0 * (5 * n * c * l + 2 * c * c * k), "flops": 4.0 * n * c * c * k * l}
    if kind == "conv":  # x, r, dy in, y, dx out
        ci, co, l, k = case["ci"], case["co"], case["l"], case["k"]
        return {"bytes": 4.0 * (n * l * (2 * ci + 3 * co) + 2 * ci * co * k), "flops": 6.0 * n * ci * co * k * l}
    if kind == "convt":
        ci, co, l, k, st = case["ci"], case["co"], case["l"], case["k"], case["s"]
        return {"bytes": 4.0 * (n * l * (2 * ci + 2 * co * st) + 2 * ci * co * k), "flops": 6.0 * n * ci * co * k * l}
    if kind == "adain":  # x, dy in, y, dx out
        return {"bytes": 16.0 * n * case["c"] * case["l"], "flops": 60.0 * n * case["c"] * case["l"]}
    if kind == "spectral":
        l, nf, hop = case["l"], CFG["n_fft"], CFG["hop"]
        return {"bytes": 4.0 * n * (2 * (nf + 2) * l + 2 * (l - 1) * hop), "flops": 300.0 * n * l}
    r, sd = config.affine_rows(CFG), CFG["style_dim"]
    return {"bytes": 4.0 * (2 * r * sd + 2 * r + 2 * n * (r + sd)), "flops": 6.0 * n * r * sd}


def tolerance(case):
    if case["kind"] in ("infer", "train", "lora"):
        # float sums through every layer, and leaky slopes that rounding picks near zero: up to 1e-5 against another
        # implementation with double sums
        return {"rel": 5e-5, "max": 1e-2}
    # one layer's float sums: up to 1.1e-6 against 64 bits, over a few thousand to half a million terms
    return {"rel": 5e-6, "max": 2e-4}


# ─── the same in 64 bits ─────────────────────────────────────────────────────


def _corr(x, w, k, stride, pad, dil):
    """conv1d of x (n, ci, l) with w (co, ci * k): one product per tap."""
    wk = w.reshape(w.shape[0], -1, k)
    x = F.pad(x, (pad, pad))
    lo = (x.shape[-1] - dil * (k - 1) - 1) // stride + 1
    y = 0
    for t in range(k):
        y = y + torch.matmul(wk[:, :, t].contiguous(), x[:, :, t * dil:t * dil + (lo - 1) * stride + 1:stride].contiguous())
    return y


def _convt(x, w, k, stride, pad):
    """conv_transpose1d of x (n, ci, l) with w (ci, co * k): each tap's product lands stride apart."""
    n, ci, l = x.shape
    wk = w.reshape(ci, -1, k)
    full = x.new_zeros(n, wk.shape[1], (l - 1) * stride + k)
    for t in range(k):
        at = slice(t, t + (l - 1) * stride + 1, stride)
        part = torch.matmul(wk[:, :, t].t().contiguous(), x)
        full = full.index_add(2, torch.arange(full.shape[2], device=x.device)[at], part)
    return full[..., pad:full.shape[2] - pad]


def _adain(x, h):
    """(1 + gamma) * instance norm + beta, (gamma, beta) the two halves of h (n, 2c)."""
    c = x.shape[1]
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (1.0 + h[:, :c, None]) * (x - m) / torch.sqrt(v + EPS) + h[:, c:, None]


def _snake(x, a):
    a = a.reshape(1, -1, 1)
    return x + torch.sin(a * x) ** 2 / a


def _istft(post):
    nf, hop = CFG["n_fft"], CFG["hop"]
    fq = nf // 2 + 1
    spec = torch.exp(post[:, :fq]) * torch.exp(1j * torch.sin(post[:, fq:]))
    win = torch.hann_window(nf, periodic=True, dtype=torch.float64, device=post.device)
    return torch.istft(spec, nf, hop, nf, window=win, center=True)


def _grads(loss, *ts):
    return [g.detach() for g in torch.autograd.grad(loss, ts)]


class _Decoder:
    """The decoder back half as a torch float64 graph, its AdaIN affines by unit name."""

    def __init__(self, params, affine):
        self.p, self.affine = params, affine

    def conv(self, name, x, k, stride=1, pad=0, dil=1):
        b = self.p.get(name + ".bias")
        y = _corr(x, self.p[name + ".weight"], k, stride, pad, dil)
        return y if b is None else y + b.reshape(1, -1, 1)

    def block(self, name, x, up):
        r = F.leaky_relu(_adain(x, self.affine[name + ".norm1"]), 0.2)
        if up:
            w, b = self.p[name + ".pool.weight"], self.p[name + ".pool.bias"].reshape(1, -1, 1)
            nxt = F.pad(r, (0, 1))[..., 1:]
            even, odd = w[None, :, 1:2] * r, w[None, :, 0:1] * nxt + w[None, :, 2:3] * r
            r = torch.stack([even, odd], -1).reshape(r.shape[0], r.shape[1], -1) + b
        r = self.conv(name + ".conv1", r, 3, pad=1)
        r = F.leaky_relu(_adain(r, self.affine[name + ".norm2"]), 0.2)
        r = self.conv(name + ".conv2", r, 3, pad=1)
        sc = torch.repeat_interleave(x, 2, -1) if up else x
        if name + ".conv1x1.weight" in self.p:
            sc = self.conv(name + ".conv1x1", sc, 1)
        return (r + sc) / math.sqrt(2.0)

    def resblock(self, name, x, k, dils):
        for i, d in enumerate(dils):
            y = _snake(_adain(x, self.affine[f"{name}.adain1.{i}"]), self.p[f"{name}.alpha1.{i}"])
            y = self.conv(f"{name}.convs1.{i}", y, k, pad=d * (k - 1) // 2, dil=d)
            y = _snake(_adain(y, self.affine[f"{name}.adain2.{i}"]), self.p[f"{name}.alpha2.{i}"])
            x = x + self.conv(f"{name}.convs2.{i}", y, k, pad=(k - 1) // 2)
        return x

    def __call__(self, asr, f0, nn, har):
        c, d = CFG, "decoder.module."
        f0, nn = (self.conv(d + m, v[:, None], 3, stride=2, pad=1) for m, v in (("F0_conv", f0), ("N_conv", nn)))
        x = self.block(d + "encode", torch.cat([asr, f0, nn], 1), False)
        asr_res, res = self.conv(d + "asr_res.0", asr, 1), True
        for i in range(c["n_decode"]):
            up = i == c["dec_up_at"]
            x = self.block(d + f"decode.{i}", torch.cat([x, asr_res, f0, nn], 1) if res else x, up)
            res = res and not up
        g = d + "generator."
        for i in range(c["n_ups"]):
            last = i + 1 == c["n_ups"]
            x = F.leaky_relu(x, 0.1)
            rest = math.prod(c["ups_rates"][i + 1:c["n_ups"]])
            src = (self.conv(g + f"noise_convs.{i}", har, 1) if last else
                   self.conv(g + f"noise_convs.{i}", har, 2 * rest, stride=rest, pad=(rest + 1) // 2))
            src = self.resblock(g + f"noise_res.{i}", src, 11 if last else 7, [1, 3, 5])
            u, k = c["ups_rates"][i], c["ups_kernels"][i]
            x = _convt(x, self.p[g + f"ups.{i}.weight"], k, u, (k - u) // 2) + self.p[g + f"ups.{i}.bias"].reshape(1, -1, 1)
            if last:
                x = torch.cat([x[..., 1:2], x], -1)  # one sample of reflection on the left
            x = x + src
            x = sum(self.resblock(g + f"resblocks.{i * c['n_kernels'] + j}", x, c["rb_kernels"][j], c["rb_dil"][j])
                    for j in range(c["n_kernels"])) / c["n_kernels"]
        k = c["conv_post_k"]
        return _istft(self.conv(g + "conv_post", F.leaky_relu(x, 0.01), k, pad=k // 2))


def _exact_lora(s):
    m, lora = s["model"], s["lora"]
    p = {name: v.double() for name, v in _param_views(m).items()}
    t = {name: _view(lora, *lora.tensor(name)).double().requires_grad_(True) for name in ("A", "B", "W1", "W2")}
    style = s["style"].double()
    gate = torch.tanh(s["cond"].double() @ t["W1"].t()) @ t["W2"].t()
    aff, r = {}, lora.rank
    for i, (name, c, off) in enumerate(m.units()):
        h = gate * (style @ t["A"][i * r:(i + 1) * r].t())
        w, b = p[name + ".fc.weight"], p[name + ".fc.bias"].reshape(1, -1)
        aff[name] = style @ w.t() + b + lora.scale * (h @ t["B"][off:off + 2 * c].t())
    audio = _Decoder(p, aff)(s["asr"].double(), s["f0"].double(), s["nn"].double(), s["har"].double())
    loss = (audio * s["daudio"].double()).sum()
    out = dict(zip(("dA", "dB", "dW1", "dW2"), _grads(loss, t["A"], t["B"], t["W1"], t["W2"])))
    return {"audio": audio.detach(), **out}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("infer", "train"):
        return None  # the harmonic source's phase is a float recurrence by definition
    s = prepare(case, seed)
    d = {k: v.double() for k, v in s.items() if isinstance(v, torch.Tensor)}
    if kind == "lora":
        return _exact_lora(s)
    if kind == "resconv_fwd":
        k, dil = case["k"], case["d"]
        y = _corr(d["x"], d["w"], k, 1, dil * (k - 1) // 2, dil) + d["b"].reshape(1, -1, 1)
        if case["res"]:
            y += d["r"]
        mean = y.mean(-1)
        var = ((y - mean[..., None]) ** 2).mean(-1)
        return {"y": y, "stats": torch.stack([mean, 1.0 / torch.sqrt(var + EPS)], -1).reshape(-1, 2)}
    if kind == "resconv_bwd":
        k, dil, c = case["k"], case["d"], case["c"]
        p = dil * (k - 1) // 2
        flip = d["w"].reshape(c, c, k).transpose(0, 1).flip(2).reshape(c, c * k)
        dact = _corr(d["dy"], flip, k, 1, dil * (k - 1) - p, dil)
        x, gb, alpha = (d[v].requires_grad_(True) for v in ("x", "gb", "alpha"))
        dx, dgb, dalpha = _grads((_snake(_adain(x, gb), alpha) * dact).sum(), x, gb, alpha)
        return {"dx": dx + d["r"], "dgb": dgb, "dw": _wgrad(d["act"], d["dy"], k, 1, p, dil), "db": d["dy"].sum((0, 2)),
                "dalpha": dalpha}
    if kind == "conv":
        ci, co, k = case["ci"], case["co"], case["k"]
        y = (_corr(d["x"], d["w"], k, 1, k // 2, 1) + d["b"].reshape(1, -1, 1) + d["r"]) * math.sqrt(0.5)
        flip = d["w"].reshape(co, ci, k).transpose(0, 1).flip(2).reshape(ci, co * k)
        return {"y": y, "dx": _corr(d["dy"], flip, k, 1, k - 1 - k // 2, 1), "dw": _wgrad(d["x"], d["dy"], k, 1, k // 2, 1),
                "db": d["dy"].sum((0, 2))}
    if kind == "convt":
        k, st = case["k"], case["s"]
        p = (k - st) // 2
        return {"y": _convt(d["x"], d["w"], k, st, p) + d["b"].reshape(1, -1, 1), "dx": _corr(d["dy"], d["w"], k, st, p, 1),
                "dw": _wgrad(d["dy"], d["x"], k, st, p, 1), "db": d["dy"].sum((0, 2))}
    if kind == "adain":
        x, gb, alpha = (d[v].requires_grad_(True) for v in ("x", "gb", "alpha"))
        y = _snake(_adain(x, gb), alpha)
        dx, dgb, dalpha = _grads((y * d["dy"]).sum(), x, gb, alpha)
        mean = x.detach().mean(-1)
        var = ((x.detach() - mean[..., None]) ** 2).mean(-1)
        return {"y": y.detach(), "stats": torch.stack([mean, 1.0 / torch.sqrt(var + EPS)], -1).reshape(-1, 2), "dx": dx,
                "dgb": dgb, "dalpha": dalpha}
    if kind == "spectral":
        post = d["post"].requires_grad_(True)
        audio = _istft(post)
        return {"audio": audio.detach(), "dpost": _grads((audio * d["da"]).sum(), post)[0]}
    return {"gb": d["style"] @ d["w"].t() + d["b"], "dstyle": d["dgb"] @ d["w"], "dw": (d["dgb"].t() @ d["style"]).reshape(-1),
            "db": d["dgb"].sum(0)}


def _wgrad(x, dy, k, stride, pad, dil):
    """dW[m, c * k + t] = sum over utterances and positions of dy[m, l] * x[c, l * stride + t * dil - pad]."""
    x = F.pad(x, (pad, pad + dil * k))
    lo, out = dy.shape[-1], []
    for t in range(k):
        xs = x[:, :, t * dil:t * dil + (lo - 1) * stride + 1:stride].contiguous()
        out.append(sum(dy[i] @ xs[i].t() for i in range(dy.shape[0])))
    return torch.stack(out, -1).reshape(-1)
