"""The framework's calls as programs make them, as cases that can be timed and compared.

Every case is one pass through a public entry point of lazylora_amd on inputs made from a seed:
the single-matrix products that a trainer calls expert by expert (`gemm`, `gemm_t`, `dequant`),
the routed-expert layer (`routed_experts_forward` / `routed_experts_backward` with a kept
workspace, or the autograd node `RoutedExpertsFunction`), the router's selection and the whole
latent MoE block. `listed()` names the cases, `draw()` makes more of the same ranges.

Weights are uniform e2m1 codes with E8M0 scales 2^-10 .. 2^-6, activations, router logits and
upstream gradients ~N(0, 1), as in bench.py.
"""
import math
import types

import torch

SCALE_LO, SCALE_HI = 117, 121  # E8M0 2^-10 .. 2^-6


# ---------------------------------------------------------------- the cases
def _routed(name, N, k, E, D, F, mode, routing="uniform", layouts="none", act="swiglu", h="f32", rank=0,
            via="calls"):
    return {"name": name, "kind": "routed", "mode": mode, "N": N, "k": k, "E": E, "D": D, "F": F, "routing": routing,
            "layouts": layouts, "act": act, "h": h, "rank": rank, "via": via}


def listed():
    return [
        # a tiny layer trained through the autograd node (config 1 of the benchmark): launches and
        # host work, hardly any data
        _routed("tiny_step", 64, 2, 8, 256, 128, "step", via="autograd"),
        # one row through one expert matrix: the reference's native.kernel().gemm for an expert that
        # one token chose
        {"name": "gemm_row1", "kind": "gemm", "M": 1, "R": 2048, "K": 7168, "x": "f32"},
        # the same call on the longer bucket of a popular expert, ragged against the 16-row tiles
        {"name": "gemm_rows200", "kind": "gemm", "M": 200, "R": 7168, "K": 2048, "x": "f32"},
        # the transposed product of the manual backward at the 22 rows per expert that the reference
        # quotes its own kernel at, in that model's expert geometry
        {"name": "gemm_t_rows22", "kind": "gemm_t", "M": 22, "R": 3072, "K": 3584, "x": "f32"},
        # widening one packed expert matrix to bf16, the reference's branch for buckets over 48 rows
        {"name": "dequant_bf16", "kind": "dequant", "R": 7168, "K": 2048, "out": "bf16"},
        # expert selection of 1024 tokens with its gradient: the router of a full batch
        {"name": "router_1024", "kind": "router", "N": 1024, "E": 896, "k": 16, "renorm": True, "scale": 2.5},
        # serving, one token at a time: the resident layer with its forward layout
        _routed("decode_1", 1, 8, 896, 7168, 2048, "forward", layouts="forward", h="bf16"),
        # prefill of long buckets: 32 experts with 256 tokens each (config 2's largest bucket)
        _routed("experts_256", 8192, 1, 32, 7168, 2048, "forward", routing="sorted", layouts="forward"),
        # a LoRA training step on a layer that is streamed through HBM (checkpoint layout only), the
        # reference model's own geometry and activation, a ragged batch
        _routed("lora_step", 1000, 16, 128, 3584, 3072, "step", act="situ", rank=16, via="autograd"),
        # the latent MoE block, forward and input gradient: router, shared expert, projections, experts
        {"name": "latent_block", "kind": "block", "N": 128, "H": 7168, "D": 3584, "F": 3072, "Ds": 3072, "E": 64,
         "k": 16},
        # a training step of the full layer under skewed routing: few, long buckets
        _routed("step_zipf", 1024, 8, 896, 7168, 2048, "step", routing="zipf", layouts="both"),
        # a training step of the full layer under uniform routing: every expert's weights once per
        # direction, the benchmark's headline
        _routed("step_uniform", 1024, 8, 896, 7168, 2048, "step", layouts="both"),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


GEOMETRIES = ((7168, 2048), (3584, 3072), (2048, 1024))


def draw(rng):
    kind = rng.choice(("gemm", "gemm_t", "dequant", "router", "small", "decode", "train", "train", "experts", "block"))
    if kind in ("gemm", "gemm_t"):
        R, K = rng.choice(((2048, 7168), (7168, 2048), (3072, 3584), (3584, 3072),
                           (_log(rng, 500, 7168), 32 * _log(rng, 16, 224))))
        return {"kind": kind, "M": _log(rng, 1, 256), "R": R, "K": K, "x": rng.choice(("f32", "f32", "bf16"))}
    if kind == "dequant":
        return {"kind": kind, "R": _log(rng, 500, 7168), "K": 32 * _log(rng, 16, 224), "out": rng.choice(("bf16", "f32"))}
    if kind == "router":
        E = _log(rng, 8, 896)
        return {"kind": kind, "N": _log(rng, 1, 1024), "E": E, "k": rng.randint(1, min(E, 16)),
                "renorm": rng.random() < 0.7, "scale": rng.choice((1.0, 2.5))}
    act, h = rng.choice(("swiglu", "situ")), rng.choice(("f32", "bf16"))
    layouts = rng.choice(("none", "forward", "both"))
    routing = rng.choice(("uniform", "zipf"))
    if kind == "small":  # layers of tests and small models: multiples of 32, on and off the layouts' own
        E = rng.randint(1, 16)
        D, F = (32 * _log(rng, 4, 64) for _ in range(2))
        return _routed("", _log(rng, 1, 300), rng.randint(1, min(E, 8)), E, D, F, "step", routing, layouts, act, h,
                       rng.choice((0, 0, 8, 16)), "autograd")
    D, F = rng.choice(GEOMETRIES)
    if kind == "decode":
        return _routed("", _log(rng, 1, 64), rng.choice((1, 2, 8, 16)), _log(rng, 16, 896), D, F, "forward", routing,
                       rng.choice(("none", "forward")), act, h)
    if kind == "train":
        return _routed("", _log(rng, 100, 1024), rng.choice((2, 8, 16)), _log(rng, 16, 256), D, F, "step", routing,
                       layouts, act, h, rng.choice((0, 0, 8, 16)), rng.choice(("calls", "autograd")))
    if kind == "experts":
        E = 32
        return _routed("", E * _log(rng, 1, 256), 1, E, D, F, "forward", "sorted", rng.choice(("none", "forward")), act, h)
    H = rng.choice((2048, 7168))
    return {"kind": "block", "N": _log(rng, 4, 256), "H": H, "D": H // 2, "F": 1024, "Ds": 1024, "E": _log(rng, 16, 64),
            "k": rng.choice((2, 8, 16))}


def _named(case):
    c = dict(case)
    c.pop("name", None)
    return c


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _codes(gen, *shape):
    n = math.prod(shape)
    words = torch.empty((n + 7) // 8, dtype=torch.int64, device="cuda").random_(-2 ** 63, None, generator=gen)
    return words.view(torch.uint8)[:n].view(shape)


def _scales(gen, *shape):
    return torch.randint(SCALE_LO, SCALE_HI + 1, shape, dtype=torch.uint8, device="cuda", generator=gen)


def _randn(gen, *shape, dtype="f32"):
    x = torch.randn(shape, device="cuda", generator=gen)
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _packed(gen, *shape):
    """Codes and scales of MXFP4 matrices [..., R, K]."""
    lead, K = shape[:-1], shape[-1]
    return _codes(gen, *lead, K // 2), _scales(gen, *lead, K // 32)


def _weights(gen, E, D, F):
    """(w1p, w1s, w3p, w3s, w2p, w2s), stacked expert-major."""
    return (*_packed(gen, E, F, D), *_packed(gen, E, F, D), *_packed(gen, E, D, F))


def _routing(gen, c):
    """(indices [N, k] int64, softmax weights [N, k] fp32)."""
    N, k, E = c["N"], c["k"], c["E"]
    if c["routing"] == "sorted":  # tokens in order of their expert, equally many each
        return (torch.arange(N, device="cuda") * E // N).reshape(N, 1), torch.ones((N, 1), device="cuda")
    logits = _randn(gen, N, E)
    if c["routing"] == "zipf":
        rank = torch.randperm(E, device="cuda", generator=gen) + 1
        logits = logits - 1.1 * torch.log(rank.float())
    val, idx = torch.topk(logits, k, dim=-1, sorted=True)
    return idx.contiguous(), torch.softmax(val.double(), dim=-1).float().contiguous()


def _adapters(gen, rank, D, F):
    if not rank:
        return None
    def one(n_in, n_out):
        return types.SimpleNamespace(lora_A=torch.nn.Parameter(0.02 * _randn(gen, rank, n_in)),
                                     lora_B=torch.nn.Parameter(0.02 * _randn(gen, n_out, rank)), scaling=32.0 / rank,
                                     dropout_rate=0.0)
    return one(D, F), one(D, F), one(F, D)


def _inputs(case, seed):
    """The tensors of a case, made from the seed alone (prepare and exact share them)."""
    c, gen = _named(case), _gen(seed)
    s = types.SimpleNamespace(c=c)
    kind = c["kind"]
    if kind in ("gemm", "gemm_t"):
        s.packed, s.scales = _packed(gen, c["R"], c["K"])
        s.x = _randn(gen, c["M"], c["K"] if kind == "gemm" else c["R"], dtype=c["x"])
    elif kind == "dequant":
        s.packed, s.scales = _packed(gen, c["R"], c["K"])
    elif kind == "router":
        s.logits = _randn(gen, c["N"], c["E"])
        s.bias = 0.1 * _randn(gen, c["E"])
        s.gw = _randn(gen, c["N"], c["k"])
    elif kind == "routed":
        s.weights = _weights(gen, c["E"], c["D"], c["F"])
        s.h = _randn(gen, c["N"], c["D"], dtype=c["h"])
        s.idx, s.w = _routing(gen, c)
        s.lora = _adapters(gen, c["rank"], c["D"], c["F"])
        s.g = _randn(gen, c["N"], c["D"]) if c["mode"] == "step" else None
    else:
        H, D, F, Ds, E = c["H"], c["D"], c["F"], c["Ds"], c["E"]
        s.weights = _weights(gen, E, D, F)
        s.dense = {"gate": _randn(gen, E, H) / math.sqrt(H), "bias": 0.1 * _randn(gen, E),
                   "w1": _randn(gen, Ds, H) / math.sqrt(H), "w3": _randn(gen, Ds, H) / math.sqrt(H),
                   "w2": _randn(gen, H, Ds) / math.sqrt(Ds), "down": _randn(gen, D, H) / math.sqrt(H),
                   "up": _randn(gen, H, D) / math.sqrt(D), "norm": 1 + 0.1 * _randn(gen, D)}
        s.x = _randn(gen, c["N"], H)
        s.g = _randn(gen, c["N"], H)
    return s


def prepare(case, seed):
    from lazylora_amd.experts import ExpertLayer
    from lazylora_amd.native import kernel

    s = _inputs(case, seed)
    c = s.c
    s.kernel = kernel()
    if s.kernel is None:
        raise RuntimeError("the native library is not available")
    if c["kind"] == "routed":
        s.layer = ExpertLayer(*s.weights)
        del s.weights
        if c["layouts"] != "none" and (c["D"] % 512 == 0 or c["F"] % 512 == 0):
            s.layer.prepare_forward_layout()
        if c["layouts"] == "both":
            s.layer.prepare_backward_layout()
        if c["via"] == "calls":
            s.ws = torch.empty(s.kernel.moe_workspace_bytes(c["N"], c["k"], c["E"], c["D"], c["F"]),
                               dtype=torch.uint8, device="cuda")
        else:
            s.h.requires_grad_()
            s.w.requires_grad_()
    elif c["kind"] == "block":
        from lazylora_amd.latent_moe import LatentMoEBlock
        d = s.dense
        s.block = LatentMoEBlock(ExpertLayer(*s.weights), d["gate"], d["bias"], d["w1"], d["w3"], d["w2"], d["down"],
                                 d["up"], d["norm"], top_k=c["k"], act="situ")
        del s.weights, s.dense
        s.x.requires_grad_()
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    c = s.c
    kind = c["kind"]
    if kind == "gemm":
        return s.kernel.gemm(s.x, s.packed, s.scales)
    if kind == "gemm_t":
        return s.kernel.gemm_t(s.x, s.packed, s.scales)
    if kind == "dequant":
        return s.kernel.dequant(s.packed, s.scales, out_dtype=torch.bfloat16 if c["out"] == "bf16" else torch.float32)
    if kind == "router":
        idx, w = s.kernel.router_topk(s.logits, s.bias, c["k"], c["scale"], c["renorm"])
        return {"idx": idx, "w": w,
                "grad_logits": s.kernel.router_topk_backward(s.logits, idx, s.gw, c["scale"], c["renorm"])}
    if kind == "block":
        out, idx, w = s.block(s.x)
        (gx,) = torch.autograd.grad(out, s.x, s.g)
        return {"out": out.detach(), "idx": idx, "w": w.detach(), "grad_x": gx}
    return _run_routed(s, c)


def _run_routed(s, c):
    from lazylora_amd.routed import RoutedExpertsFunction, routed_experts_backward, routed_experts_forward

    step = c["mode"] == "step"
    if s.lora:  # optimizer.zero_grad(set_to_none=True)
        for m in s.lora:
            m.lora_A.grad = m.lora_B.grad = None
    if c["via"] == "autograd":
        out = RoutedExpertsFunction.apply(s.h, s.w, s.idx, s.layer, c["act"], None, s.lora)
        gh, gw = torch.autograd.grad(out, (s.h, s.w), s.g)
        out = out.detach()
    else:
        out = routed_experts_forward(s.h, s.idx, s.w, s.layer, act=c["act"], save_for_backward=step, workspace=s.ws,
                                     lora=s.lora)
        if not step:
            return {"out": out}
        gh, gw = routed_experts_backward(s.h, s.idx, s.w, s.layer, s.g, act=c["act"], reuse_forward=True,
                                         workspace=s.ws, lora=s.lora)
    res = {"out": out, "grad_h": gh, "grad_w": gw}
    if s.lora:
        for n, m in zip(("gate", "up", "down"), s.lora):
            res[n + "_A"], res[n + "_B"] = m.lora_A.grad, m.lora_B.grad
    return res


# ---------------------------------------------------------------- what a pass cannot do without
def _mx_bytes(R, K):
    return R * K // 2 + R * K // 32


def _active(c):
    """Experts that a routing of this kind selects (uniform: expected distinct; zipf: the share that
    the benchmark's skewed routing of this many pairs reaches, about a seventh)."""
    N, k, E = c["N"], c["k"], c["E"]
    if c["routing"] == "sorted":
        return min(E, N)
    uniform = E * (1.0 - (1.0 - min(1.0, k / E)) ** N)
    return min(uniform, max(k, 0.134 * E)) if c["routing"] == "zipf" else uniform


def work(case):
    c = _named(case)
    kind = c["kind"]
    if kind in ("gemm", "gemm_t"):
        M, R, K = c["M"], c["R"], c["K"]
        x = 2 if c["x"] == "bf16" else 4
        n_in, n_out = (K, R) if kind == "gemm" else (R, K)
        return {"bytes": _mx_bytes(R, K) + x * M * n_in + 4 * M * n_out, "flops": 2 * M * R * K}
    if kind == "dequant":
        return {"bytes": _mx_bytes(c["R"], c["K"]) + (2 if c["out"] == "bf16" else 4) * c["R"] * c["K"], "flops": 0}
    if kind == "router":
        N, E, k = c["N"], c["E"], c["k"]
        return {"bytes": 4 * N * E * 2 + 4 * E + N * k * (8 + 4 + 4), "flops": 0}
    if kind == "block":
        N, H, D, F, Ds, E, k = (c[n] for n in ("N", "H", "D", "F", "Ds", "E", "k"))
        act = E * (1.0 - (1.0 - k / E) ** N)
        dense = E * H + 3 * Ds * H + 2 * D * H
        return {"bytes": int(2 * act * 3 * _mx_bytes(D, F) + 4 * dense + 4 * N * H * 4),
                "flops": 2 * (2 * N * dense + 6 * N * k * D * F)}
    N, k, E, D, F, r = (c[n] for n in ("N", "k", "E", "D", "F", "rank"))
    passes = 2 if c["mode"] == "step" else 1
    h = 2 if c["h"] == "bf16" else 4
    io = N * D * (h + 4) + N * k * 12
    if passes == 2:
        io += N * D * (4 + h) + N * k * 4 + 2 * 4 * r * 3 * (D + F)
    return {"bytes": int(passes * _active(c) * 3 * _mx_bytes(D, F)) + io,
            "flops": passes * (6 * N * k * D * F + (6 * N * k * r * (D + F) if r else 0))}


def tolerance(case):
    """Measured on the first version of the kernels against 64 bits, times about four."""
    c = _named(case)
    kind = c["kind"]
    if kind == "gemm":
        # activations to two 4-bit-mantissa terms (about 8 significant bits): 6e-4
        return {"rel": 2.5e-3, "max": 2e-2}
    if kind == "gemm_t":
        # bf16 hi + lo gradients (about 16 significant bits): 3e-6
        return {"rel": 1e-5, "max": 2e-4}
    if kind == "dequant":
        return "exact"
    if kind == "router":
        # fp32 throughout (8e-8); two scores a last bit apart can change places
        return {"rel": 2e-6, "max": 1e-3, "differ": 1e-3}
    if kind == "block":
        # the router's selection of a token can turn on the last bit of an fp32 logit
        # (out 9.7e-4)
        return {"rel": 4e-3, "max": 5e-2, "differ": 2e-3}
    # routed layer: two such products in a row (1.1e-3) and, in a step, the transposed ones after
    # them; bf16 activations round their gradient to bf16 (1.7e-3)
    return {"rel": 7e-3 if c["h"] == "bf16" and c["mode"] == "step" else 4.5e-3, "max": 5e-2}


# ---------------------------------------------------------------- 64-bit reference
_LUT = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _dense(packed, scales):
    """W [R, K] in float64 from codes [R, K/2] and scales [R, K/32] (all below 253 here)."""
    lut = torch.tensor(_LUT, dtype=torch.float64, device=packed.device)
    pairs = torch.stack((lut.repeat(16), lut.repeat_interleave(16)), dim=-1)  # byte -> (low, high nibble)
    R, Kh = packed.shape
    w = pairs[packed.int()].view(R, Kh // 16, 32)
    return (w * torch.exp2(scales.double() - 127).unsqueeze(-1)).view(R, Kh * 2)


def _glu(g, u, act):
    if act == "swiglu":
        return g * torch.sigmoid(g) * u
    return 4.0 * torch.tanh(g / 4.0) * torch.sigmoid(g) * (25.0 * torch.tanh(u / 25.0))


def _experts64(h, idx, w, weights, act, lora):
    """The routed sum of h [N, D] in float64, differentiable by autograd in h, w and the adapters
    (given as float64 (A, B, scaling) triples)."""
    out = torch.zeros(h.shape, dtype=torch.float64, device=h.device)
    for e in torch.unique(idx).tolist():
        t, slot = torch.nonzero(idx == e, as_tuple=True)
        out = _Expert64.apply(out, h, w, t, slot, weights, e, act, lora, *([p for m in lora for p in m[:2]] if lora else ()))
    return out


class _Expert64(torch.autograd.Function):
    """out + one expert's weighted rows; the dense float64 weights live only inside each call."""

    @staticmethod
    def _rows(x, wt, weights, e, act, lora):
        lin = lambda v, p, s, m: v @ _dense(p[e], s[e]).T + (m[2] * (v @ m[0].T) @ m[1].T if m else 0.0)
        w1p, w1s, w3p, w3s, w2p, w2s = weights
        gate_m, up_m, down_m = lora if lora else (None, None, None)
        a = _glu(lin(x, w1p, w1s, gate_m), lin(x, w3p, w3s, up_m), act)
        return lin(a, w2p, w2s, down_m) * wt.unsqueeze(1)

    @staticmethod
    def forward(ctx, out, h, w, t, slot, weights, e, act, lora, *params):
        ctx.save_for_backward(h, w, t, slot, *params)
        ctx.weights, ctx.e, ctx.act, ctx.lora = weights, e, act, lora
        return out.index_add(0, t, _Expert64._rows(h[t], w[t, slot], weights, e, act, lora))

    @staticmethod
    def backward(ctx, g):
        h, w, t, slot, *params = ctx.saved_tensors
        x, wt = h[t].detach().requires_grad_(), w[t, slot].detach().requires_grad_()
        ps = [p.detach().requires_grad_() for p in params]
        lora = [(ps[2 * i], ps[2 * i + 1], m[2]) for i, m in enumerate(ctx.lora)] if ctx.lora else None
        with torch.enable_grad():
            rows = _Expert64._rows(x, wt, ctx.weights, ctx.e, ctx.act, lora)
        gx, gwt, *gp = torch.autograd.grad(rows, (x, wt, *ps), g[t])
        gh = torch.zeros_like(h).index_add_(0, t, gx)
        gw = torch.zeros_like(w)
        gw[t, slot] = gwt
        return (g, gh, gw, None, None, None, None, None, None, *gp)


def exact(case, seed):
    s = _inputs(case, seed)
    c = s.c
    kind = c["kind"]
    if kind == "gemm":
        return s.x.double() @ _dense(s.packed, s.scales).T
    if kind == "gemm_t":
        return s.x.double() @ _dense(s.packed, s.scales)
    if kind == "dequant":
        return _dense(s.packed, s.scales)
    if kind == "router":
        lg = s.logits.double().requires_grad_()
        idx, w = _select64(lg, s.bias.double(), c["k"], c["scale"], c["renorm"])
        (gl,) = torch.autograd.grad(w, lg, s.gw.double())
        return {"idx": idx, "w": w.detach(), "grad_logits": gl}
    if kind == "block":
        d = {n: v.double() for n, v in s.dense.items()}
        x = s.x.double().requires_grad_()
        idx, w = _select64(x @ d["gate"].T, d["bias"], c["k"], 1.0, True)
        shared = _glu(x @ d["w1"].T, x @ d["w3"].T, "situ") @ d["w2"].T
        routed = _experts64(x @ d["down"].T, idx, w, s.weights, "situ", None)
        routed = routed * torch.rsqrt(routed.pow(2).mean(-1, keepdim=True) + 1e-5) * d["norm"]
        out = shared + routed @ d["up"].T
        (gx,) = torch.autograd.grad(out, x, s.g.double())
        return {"out": out.detach(), "idx": idx, "w": w.detach(), "grad_x": gx}
    step = c["mode"] == "step"
    h, w = s.h.double().requires_grad_(step), s.w.double().requires_grad_(step)
    lora = [(m.lora_A.detach().double().requires_grad_(step), m.lora_B.detach().double().requires_grad_(step), m.scaling)
            for m in s.lora] if s.lora else None
    out = _experts64(h, s.idx, w, s.weights, c["act"], lora)
    if not step:
        return {"out": out}
    params = [p for m in lora for p in m[:2]] if lora else []
    gh, gw, *gp = torch.autograd.grad(out, (h, w, *params), s.g.double())
    res = {"out": out.detach(), "grad_h": gh, "grad_w": gw}
    for i, n in enumerate(("gate", "up", "down") if lora else ()):
        res[n + "_A"], res[n + "_B"] = gp[2 * i], gp[2 * i + 1]
    return res


def _select64(logits, bias, k, scale, renorm):
    scores = torch.sigmoid(logits)
    idx = torch.topk(scores + bias, k, dim=-1, sorted=True).indices
    w = scores.gather(1, idx)
    if renorm and k > 1:
        w = w / (w.sum(-1, keepdim=True) + 1e-20)
    return idx, w * scale
