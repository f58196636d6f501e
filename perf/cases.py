"""The framework's work in a training program, as cases that can be timed and checked one by one.

Four entry points carry it: ``Muon.step`` (momentum, norm, Newton-Schulz, weight update and the
AdamW of the remaining parameters), the stand-alone Newton-Schulz functions, the symmetric-product
seam ``syrk_or_cublas``, and the bandwidth-bound ``Muon.clip_grad_norm_`` /
``clip_grad_norm_buckets_`` and ``fused_adamw_``. A case names the entry point (``kind``), its
sizes and its options; shapes are written ``"4*512x2048 1000x300"``.
"""
from __future__ import annotations

import math

import torch
from torch import nn

import dmuon_amd as dmuon
from dmuon_amd.optim import syrk_or_cublas

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
LR, MU, WD, EPS = 0.02, 0.95, 0.1, 1e-7
ADAMW = dict(lr=1e-3, betas=(0.9, 0.999), weight_decay=0.01, eps=1e-8)
ADAMW_STEP = 100                       # steps the AdamW state has behind it
SYRK_BC = (-4.7750, 2.0315)            # Z = b R + c R R^T


def listed():
    layer = "8*4096x4096 8*1024x4096 8*14336x4096 4*4096x14336"
    return [
        # the smallest call: one small matrix through the stand-alone function
        dict(name="ns_128x512", kind="ns", shapes="128x512", dtype="fp32", backend="gram"),
        # the reference's example training loop: 4 blocks of 512 / 2048, fp32, its head on AdamW
        dict(name="step_example_model", kind="step", shapes="8*2048x512 4*512x2048", dtype="fp32",
             master="param", backend="gram", rest="512"),
        # one 1024^2 fp32 weight, the direct form
        dict(name="step_1024x1024_direct", kind="step", shapes="1024x1024", dtype="fp32",
             master="param", backend="direct", rest=""),
        # odd and ragged weights under the default policy: fp32 masters, bf16 forward copies
        dict(name="step_ragged", kind="step", shapes="1000x300 130x250 1100x1900 2*333x1025",
             dtype="bf16", master="fp32", backend="gram", rest="1000 333"),
        # one long matrix, stored tall, fp32 master and bf16 forward copy
        dict(name="step_16384x1024", kind="step", shapes="16384x1024", dtype="bf16",
             master="fp32", backend="gram", rest=""),
        # one square matrix, updated in place
        dict(name="step_4096x4096", kind="step", shapes="4096x4096", dtype="bf16",
             master="param", backend="gram", rest=""),
        # 128 experts of one layer in two stacked weights
        dict(name="step_moe_experts", kind="step", shapes="64*1408x2048 64*2048x1408",
             dtype="bf16", master="param", backend="gram", rest="", stacked=True),
        # four transformer layers of the Llama-3-8B sizes with their norms and the embedding
        dict(name="step_four_layers", kind="step", shapes=layer, dtype="bf16", master="param",
             backend="gram", rest="9*4096 128256x4096"),
        # the stand-alone orthogonalisation of a mid-sized weight
        dict(name="ns_2048x8192", kind="ns", shapes="2048x8192", dtype="bf16", backend="gram"),
        # the symmetric products of the reference's own Newton-Schulz code on a ragged operand
        dict(name="syrk_1000x3000", kind="syrk", M=1000, K=3000, batch=1, dtype="fp16"),
        # the gradients of one transformer layer, clipped before the step
        dict(name="clip_one_layer", kind="clip", buckets=False, dtype="bf16",
             shapes="2*4096x4096 2*1024x4096 2*14336x4096 4096x14336"),
        # the norm vectors of a 32-layer model
        dict(name="adamw_norms", kind="adamw", shapes="65*4096", dtype="bf16", grad_dtype="bf16",
             stacked=True),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def side(lo, hi):                  # a third of the sides are whatever they are
        v = log_int(lo, hi)
        return v if rng.random() < 0.35 else max(64, v // 64 * 64)

    def matrix(lo, hi, most):
        m = side(lo, hi)
        n = min(most, max(m, side(m, 16 * m)))
        return (m, n) if rng.random() < 0.5 else (n, m)

    kind = rng.choice(("step",) * 5 + ("ns",) * 2 + ("syrk",) * 2 + ("clip", "adamw"))
    if kind == "step":
        shapes, flops, room = [], 0.0, 16   # a case gives back a few dozen tensors
        for _ in range(rng.choice((1, 1, 1, 2, 3, 4))):
            shape = matrix(128, 4096, 16384)
            copies = min(room, log_int(1, 12))
            while copies and flops + copies * _ns_flops(*shape, "gram") > 2e13:
                copies //= 2
            if copies:
                flops += copies * _ns_flops(*shape, "gram")
                shapes.append("%d*%dx%d" % (copies, *shape))
                room -= copies
        rest = " ".join(str(side(64, 8192)) for _ in range(rng.randrange(0, 4)))
        return dict(kind="step", shapes=" ".join(shapes), dtype=rng.choice(("fp32", "bf16")),
                    master=rng.choice(("param", "fp32")),
                    backend=rng.choice(("gram", "gram", "direct")), rest=rest)
    if kind == "ns":
        r, c = matrix(64, 2048, 8192)
        return dict(kind="ns", shapes="%d*%dx%d" % (rng.choice((1, 1, 2, 8)), r, c),
                    dtype=rng.choice(("fp32", "bf16")),
                    backend=rng.choice(("gram", "gram", "direct")))
    if kind == "syrk":
        return dict(kind="syrk", M=side(128, 4096), K=side(128, 16384), batch=rng.choice((1, 1, 4)),
                    dtype=rng.choice(("fp16", "bf16")))
    if kind == "clip":
        shapes = " ".join("%dx%d" % matrix(64, 4096, 16384) for _ in range(log_int(1, 24)))
        return dict(kind="clip", buckets=rng.random() < 0.5, shapes=shapes,
                    dtype=rng.choice(("fp32", "bf16")))
    shapes = " ".join(str(log_int(64, 1 << 22)) for _ in range(log_int(1, 16)))
    dtype = rng.choice(("fp32", "bf16"))
    return dict(kind="adamw", shapes=shapes, dtype=dtype,
                grad_dtype=rng.choice((dtype, "bf16")))


# ------------------------------------------------------------------------------------ sizes
def _shapes(text):
    out = []
    for word in text.split():
        copies, _, dims = word.rpartition("*")
        out += [tuple(int(d) for d in dims.split("x"))] * int(copies or 1)
    return out


def _ns_flops(rows, cols, backend):
    """Products of five steps, one triangle of the symmetric ones (gram: a restart at step 2)."""
    m, n = float(min(rows, cols)), float(max(rows, cols))
    sq, gram, full = m * (m + 1) * m, m * (m + 1) * n, 2 * m * m * n
    if backend == "direct":
        return 5 * (gram + sq + full)
    return 2 * (gram + full) + 5 * sq + 3 * 2 * m ** 3 + 6 * sq


def _width(dtype):
    return 4 if dtype == "fp32" else 2


def work(case):
    numels = [math.prod(s) for s in _shapes(case.get("shapes", ""))]
    total = sum(numels)
    w = _width(case["dtype"])
    if case["kind"] == "step":
        rest = sum(math.prod(s) for s in _shapes(case["rest"]))
        separate = case["master"] == "fp32" and case["dtype"] != "fp32"
        # gradient, momentum in and out, weight in and out, the forward copy
        per = w + 8 + (8 + w if separate else 2 * w)
        return {"bytes": total * per + rest * 7 * w,
                "flops": sum(_ns_flops(*s, case["backend"]) for s in _shapes(case["shapes"]))}
    if case["kind"] == "ns":
        return {"bytes": total * 2 * w,
                "flops": sum(_ns_flops(*s, case["backend"]) for s in _shapes(case["shapes"]))}
    if case["kind"] == "syrk":
        M, K, L = case["M"], case["K"], case["batch"]
        return {"bytes": L * (M * K + 2 * M * M) * w, "flops": float(L) * M * (M + 1) * (K + M)}
    if case["kind"] == "clip":
        return {"bytes": total * 2 * w, "flops": 3.0 * total}
    return {"bytes": total * (6 * w + _width(case["grad_dtype"])), "flops": 15.0 * total}


# ----------------------------------------------------------------------------------- inputs
class _Model(nn.Module):
    def __init__(self, mats, rest):
        super().__init__()
        self.mats = nn.ParameterList([nn.Parameter(t) for t in mats])
        self.rest = nn.ParameterList([nn.Parameter(t) for t in rest])


def _tensors(text, stacked, make):
    """The tensors of ``text``: one allocation each, or each run of one shape stacked in one (the
    experts' weights, a model's norms in one buffer). Returns (allocations, tensors)."""
    if not stacked:
        each = [make(s) for s in _shapes(text)]
        return each, each
    runs = [_shapes(word) for word in text.split()]
    bases = [make((len(run), *run[0])) for run in runs]
    return bases, [t for base in bases for t in base.unbind(0)]


def _ns_backend(backend):
    if backend == "direct":
        return dmuon.NewtonSchulz("direct", coefficients=dmuon.KELLER_COEFFICIENTS)
    return dmuon.NewtonSchulz("gram")


def _coefficients(backend):
    return dmuon.KELLER_COEFFICIENTS if backend == "direct" else dmuon.POLAR_EXPRESS_COEFFICIENTS


def _inputs(case, seed):
    """Every tensor of the case, from its seed: {"name": (allocations, tensors)}."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(dtype, std=0.02):
        return lambda shape: torch.empty(shape, device=DEV, dtype=dtype).normal_(
            0.0, std, generator=gen)

    def adamw(text, stacked, grad_dtype):
        return {"p": _tensors(text, stacked, normal(dtype)),
                "g": _tensors(text, False, normal(grad_dtype)),
                "m": _tensors(text, stacked, normal(dtype, 0.005)),
                "v": _tensors(text, stacked, lambda s: normal(dtype)(s).square_())}

    if case["kind"] == "syrk":
        M, K, L = case["M"], case["K"], case["batch"]
        lead = (L,) if L > 1 else ()
        X = normal(torch.float32, 1.0 / math.sqrt(K))(lead + (M, K)).to(dtype)
        return {"X": X, "R": X.new_empty(lead + (M, M)), "Z": X.new_empty(lead + (M, M))}
    stacked = case.get("stacked", False)
    if case["kind"] == "adamw":
        return adamw(case["shapes"], stacked, DTYPES[case["grad_dtype"]])
    found = {"grad": _tensors(case["shapes"], False, normal(dtype))}
    if case["kind"] == "step":
        found["weight"] = _tensors(case["shapes"], stacked, normal(dtype))
        found["momentum"] = _tensors(case["shapes"], stacked, normal(torch.float32))
        found["rest"] = adamw(case["rest"], stacked or "*" in case["rest"], dtype)
    return found


def prepare(case, seed):
    kind, t = case["kind"], _inputs(case, seed)
    if kind == "step":
        rest = t["rest"]
        model = _Model(t["weight"][1], rest["p"][1])
        dmuon.dedicate_params(model, None, lambda name, p: name.startswith("mats"), param_policy={
            "defaults": {"master_dtype": torch.float32 if case["master"] == "fp32"
                         else DTYPES[case["dtype"]]}})
        dmuon.replicate(model)
        opt = dmuon.Muon(model, lr=LR, momentum=MU, weight_decay=WD,
                         ns_backend=_ns_backend(case["backend"]), adamw_lr=ADAMW["lr"],
                         adamw_betas=ADAMW["betas"], adamw_weight_decay=ADAMW["weight_decay"],
                         adamw_eps=ADAMW["eps"])
        # the state of a program that has run some steps
        owned = dmuon.get_owned_params(model)
        for dp, grad, buf in zip(owned, t["grad"][1], t["momentum"][1]):
            dp.param.grad = grad
            opt.state[id(dp)]["momentum_buffer"] = buf
        for p, grad, m, v in zip(model.rest, rest["g"][1], rest["m"][1], rest["v"][1]):
            p.grad = grad
            opt.state[p].update(step=ADAMW_STEP, exp_avg=m, exp_avg_sq=v)
        out = {"weight": t["weight"][0], "momentum": t["momentum"][0],
               "adamw": [rest[k][0] for k in "pmv"]}
        if owned[0].publish_target() is not None:
            out["master"] = [dp._owned_data for dp in owned]
        return {"kind": kind, "opt": opt, "out": out}
    if kind == "ns":
        return {"kind": kind, "backend": case["backend"], "G": t["grad"][1]}
    if kind == "syrk":
        return {"kind": kind, **t}
    if kind == "adamw":
        return {"kind": kind, "step": ADAMW_STEP, "args": [t[k][1] for k in "pgmv"],
                "out": [t[k][0] for k in "pmv"]}
    grads = t["grad"][1]
    if case["buckets"]:
        cut = (len(grads) + 1) // 2
        return {"kind": kind, "grads": grads, "buckets": (
            dmuon.GradClipBucket("regular", grads[:cut], reduce=False),
            dmuon.GradClipBucket("muon", grads[cut:]))}
    model = _Model([torch.empty_like(g) for g in grads], [])
    dmuon.dedicate_params(model, None, lambda name, p: True)
    opt = dmuon.Muon(model)
    for p, g in zip(model.mats, grads):
        p.grad = g
    return {"kind": kind, "grads": grads, "opt": opt}


# -------------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "step":
        state["opt"].step()
        return state["out"]
    if kind == "ns":
        G = state["G"]
        if len(G) > 1:
            return dmuon.newton_schulz_batched(
                G, _coefficients(state["backend"]), backend=state["backend"],
                restart_iterations=(2,) if state["backend"] == "gram" else ())
        if state["backend"] == "gram":
            return dmuon.gram_newton_schulz(G[0])
        return dmuon.direct_newton_schulz(G[0], coefficients=dmuon.KELLER_COEFFICIENTS)
    if kind == "syrk":
        X, R, Z = state["X"], state["R"], state["Z"]
        b, c = SYRK_BC
        syrk_or_cublas(X, R)
        syrk_or_cublas(R, Z, C=R, alpha=c, beta=b)
        return [R, Z]
    if kind == "clip":
        if "buckets" in state:
            res = dmuon.clip_grad_norm_buckets_(state["buckets"], 1.0)
            norms = [s.total_norm for s in res.bucket_stats]
        else:
            norms = [state["opt"].clip_grad_norm_(1.0).total_norm]
        return {"grads": state["grads"], "norms": norms}
    state["step"] += 1
    dmuon.fused_adamw_(*state["args"], step=state["step"], **ADAMW)
    return state["out"]


# ------------------------------------------------------------------------ exact and tolerance
def _ns_exact(G, backend):
    """The composition of the five polynomials on G / (||G|| + eps), in float64."""
    X = G.double()
    X = X / (X.norm() + EPS)
    tall = X.shape[0] > X.shape[1]
    X = X.t().contiguous() if tall else X
    for a, b, c in _coefficients(backend):
        A = X @ X.t()
        X = a * X + (b * A + c * (A @ A)) @ X
    return X.t() if tall else X


def _adamw_exact(t):
    b1, b2 = ADAMW["betas"]
    step = ADAMW_STEP + 1
    new = {"p": [], "m": [], "v": []}
    for p, g, m, v in zip(*(t[k][1] for k in "pgmv")):
        p, g, m, v = (x.double() for x in (p, g, m, v))
        m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
        d = (v / (1 - b2 ** step)).sqrt() + ADAMW["eps"]
        new["p"].append(p * (1 - ADAMW["lr"] * ADAMW["weight_decay"])
                        - ADAMW["lr"] / (1 - b1 ** step) * m / d)
        new["m"].append(m)
        new["v"].append(v)
    return [_packed(new[k], t[k][0]) for k in "pmv"]


def _packed(values, allocations):
    """``values`` laid out as the allocations that hold them."""
    out, it = [], iter(values)
    for a in allocations:
        first = next(it)
        if first.numel() == a.numel():
            out.append(first.reshape(a.shape))
        else:
            out.append(torch.stack([first] + [next(it) for _ in range(a.shape[0] - 1)]))
    return out


def exact(case, seed):
    kind, t = case["kind"], _inputs(case, seed)
    if kind == "step":
        weights, bufs = [], []
        for w, g, buf in zip(t["weight"][1], t["grad"][1], t["momentum"][1]):
            buf = buf.double() * MU + g.double()
            u = _ns_exact(g.double() + MU * buf, case["backend"])
            weights.append(w.double() * (1 - LR * WD) - LR * 0.2 * math.sqrt(max(w.shape)) * u)
            bufs.append(buf)
        out = {"weight": _packed(weights, t["weight"][0]),
               "momentum": _packed(bufs, t["momentum"][0]), "adamw": _adamw_exact(t["rest"])}
        if case["master"] == "fp32" and case["dtype"] != "fp32":
            out["master"] = weights
        return out
    if kind == "ns":
        outs = [_ns_exact(G, case["backend"]) for G in t["grad"][1]]
        return outs if len(outs) > 1 else outs[0]
    if kind == "syrk":
        X, (b, c) = t["X"].double(), SYRK_BC
        R = X @ X.transpose(-1, -2).contiguous()
        return [R, c * (R @ R.transpose(-1, -2).contiguous()) + b * R]
    if kind == "adamw":
        return _adamw_exact(t)
    grads = t["grad"][1]
    cut = (len(grads) + 1) // 2
    new, norms = [], []
    for seg in ([grads[:cut], grads[cut:]] if case["buckets"] else [grads]):
        norm = math.sqrt(sum(float(g.double().square().sum()) for g in seg))
        norms.append(norm)
        new += [g.double() * min(1.0, 1.0 / (norm + 1e-6)) for g in seg]
    return {"grads": new, "norms": [torch.tensor(n, dtype=torch.float64) for n in norms]}


def tolerance(case):
    """Relative errors a few times those seen against :func:`exact`."""
    if case["kind"] == "step":
        # bf16 weights round at 2^-9; in fp32 the fp16 products' error in U shows, weighed by the
        # update's share of the weight
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3, "max": 0.2}
    if case["kind"] == "ns":
        return {"rel": 1.2e-2, "max": 0.2}      # fp16 products, five steps deep
    if case["kind"] == "syrk":
        return {"rel": 2e-3 if case["dtype"] == "fp16" else 1e-2, "max": 0.1}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.05}
    return {"rel": 2e-5, "max": 1e-4}           # 32-bit sums and element-wise arithmetic
