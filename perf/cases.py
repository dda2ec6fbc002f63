"""Workloads of the MuonAdamW optimizer, for timing and for comparing results.

A case is one call that a training program makes: a whole optimizer step over
a model's parameters (``MuonAdamW``), one branch of it (``HipMuon``,
``HipAdamW``), or one of the standalone functions (``muon_step``,
``newton_shultz_step``, ``solve_ns_kernel_1``).  ``prepare`` builds what such a
program holds before the call (parameters with gradients, the optimizer and its
state as after some steps of training), ``run`` makes the call, ``exact`` gives
the same result in float64 with plain torch.

Parameters, gradients and optimizer state are views into one flat buffer each,
as programs keep them that bucket gradients or checkpoint flat state; ``run``
returns those buffers whole.  Parameters are N(0, 0.02), gradients N(0, 1e-3),
prior momentum N(0, 1e-3), first moments N(0, 1e-4) and second moments
|N(0, 1e-6)|, as in the benchmark's configurations.
"""

import math
import sys
from pathlib import Path

import torch
import torch.nn as nn

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT / "triton-muonadamw_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "triton-muonadamw_amd"))

COEFFS = (3.4445, -4.7750, 2.0315)
MUON = {"lr": 0.02, "beta": 0.95, "eps": 1e-7, "weight_decay": 0.1, "coeffs": COEFFS, "nesterov": True, "ns_steps": 5}
ADAM = {"lr": 3e-4, "betas": (0.9, 0.95), "eps": 1e-8, "weight_decay": 0.1}
PRIOR_STEPS = 9  # the moments are those of a run that has taken this many steps


def listed():
    return [
        # The smallest whole step: the two-layer MLP of the benchmark, fp32. Latency and launches.
        {"name": "toy_mlp", "kind": "mlp", "dims": "512-2048-512", "dtype": "fp32", "amp": False},
        # A small classifier with sizes that nothing divides, a ten-row output matrix among them.
        {"name": "odd_mlp", "kind": "mlp", "dims": "785-1003-517-10", "dtype": "fp32", "amp": False},
        # The LayerNorm MLP of the hybrid benchmark: four matrices, no two of one shape class.
        {"name": "hybrid_mlp", "kind": "mlp", "dims": "1024-2048-4096-4096-1024", "dtype": "fp32", "amp": False},
        # A whole step of the GPT-2-124M set: 48 matrices in three shape classes, tied embedding, biases, norms.
        {"name": "gpt2", "kind": "gpt", "layers": 12, "d": 768, "vocab": 50257, "ctx": 1024, "dtype": "fp32"},
        # One decoder layer of the Llama-8B set with a layer's share of embedding and head, in bf16 as it is trained.
        {"name": "llama_layer_bf16", "kind": "llama", "layers": 1, "d": 4096, "kv": 1024, "ffn": 14336, "vocab": 4008,
         "dtype": "bf16"},
        # The largest launch group of the Llama-8B step: 32 gate/up matrices (14336 x 4096, the transposed path).
        {"name": "muon_gate_up_x32", "kind": "muon", "count": 32, "rows": 14336, "cols": 4096, "dtype": "fp32"},
        # Every k/v projection of the Llama-8B step: many matrices of middling size.
        {"name": "muon_kv_x64", "kind": "muon", "count": 64, "rows": 1024, "cols": 4096, "dtype": "fp32"},
        # The function for one matrix, with its orthogonalised update returned: a GPT-2 MLP matrix.
        {"name": "muon_step_one", "kind": "muon_step", "rows": 3072, "cols": 768},
        # One Newton-Schulz iteration of a bf16 matrix, as custom optimizers call it.
        {"name": "ns_iteration", "kind": "ns_step", "rows": 1024, "cols": 4096},
        # The Gram matrix of a bf16 matrix whose sizes nothing divides.
        {"name": "ns_gram_odd", "kind": "ns_gram", "rows": 1531, "cols": 3001},
        # The AdamW benchmark: 256 tensors from 1e3 to 4e6 elements in one step.
        {"name": "adamw_256_tensors", "kind": "adamw", "tensors": 256, "smallest": 1000, "largest": 4_000_000,
         "total": 1 << 26, "packed": False, "dtype": "fp32"},
        # The embedding of the Llama-8B set in bf16, the largest single AdamW tensor.
        {"name": "adamw_embedding_bf16", "kind": "adamw", "tensors": 1, "smallest": 128256 * 4096,
         "largest": 128256 * 4096, "total": 128256 * 4096, "packed": False, "dtype": "bf16"},
    ]


def draw(rng):
    def size(lo, hi):
        """Log-uniform in [lo, hi]; half of the draws rounded to a multiple of 64 where that fits."""
        x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return max(64, x // 64 * 64) if x >= 64 and rng.random() < 0.5 else x

    kind = rng.choice(["mlp", "gpt", "llama", "muon", "muon", "muon_step", "ns_step", "ns_gram", "adamw", "adamw"])
    dtype = rng.choice(["fp32", "fp32", "bf16"])
    if kind == "mlp":
        dims = [size(10, 4096) for _ in range(rng.randint(3, 5))]
        return {"kind": "mlp", "dims": "-".join(map(str, dims)), "dtype": dtype, "amp": rng.random() < 0.3}
    if kind == "gpt":
        return {"kind": "gpt", "layers": rng.randint(1, 12), "d": 64 * rng.randint(2, 16),
                "vocab": rng.randint(1000, 50257), "ctx": rng.choice([256, 512, 1024]), "dtype": dtype}
    if kind == "llama":
        heads = rng.randint(4, 32)
        return {"kind": "llama", "layers": rng.randint(1, 2), "d": 128 * heads, "kv": 128 * max(1, heads // 4),
                "ffn": 64 * int(heads * rng.uniform(5.0, 7.0)), "vocab": rng.randint(1000, 4008), "dtype": dtype}
    if kind == "muon":
        rows, cols = size(16, 14336), size(64, 4096)
        most = max(1, min(64, int(32 * 14336 * 4096 ** 2 / (max(rows, cols) * min(rows, cols) ** 2)),
                          int(1.8e9 / (rows * cols))))
        return {"kind": "muon", "count": rng.randint(1, most), "rows": rows, "cols": cols, "dtype": dtype}
    if kind in ("muon_step", "ns_step", "ns_gram"):
        rows, cols = size(64, 4096), size(64, 8192)
        return {"kind": kind, "rows": rows, "cols": cols}
    tensors = max(1, int(math.exp(rng.uniform(0.0, math.log(512)))))
    smallest = size(64, 4096)
    largest = size(8192, 4_000_000)
    return {"kind": "adamw", "tensors": tensors, "smallest": smallest, "largest": largest, "total": 0,
            "packed": rng.random() < 0.3, "dtype": dtype}


# ---------------------------------------------------------------------------
# Layouts: [(shape, branch)] in the order of the flat buffers.

def _layout(case):
    kind, out = case["kind"], []
    if kind == "mlp":  # Linear (+ LayerNorm between the layers), torch's (out, in) weights
        dims = [int(d) for d in case["dims"].split("-")]
        for i, (fi, fo) in enumerate(zip(dims[:-1], dims[1:])):
            out += [((fo, fi), "muon"), ((fo,), "adam")]
            if i < len(dims) - 2:
                out += [((fo,), "adam"), ((fo,), "adam")]
    elif kind == "gpt":  # Conv1D weights (in, out); tied head
        d = case["d"]
        out = [((case["vocab"], d), "adam"), ((case["ctx"], d), "adam")]
        for _ in range(case["layers"]):
            out += [((d,), "adam"), ((d,), "adam"), ((d, 3 * d), "muon"), ((3 * d,), "adam"), ((d, d), "muon"),
                    ((d,), "adam"), ((d,), "adam"), ((d,), "adam"), ((d, 4 * d), "muon"), ((4 * d,), "adam"),
                    ((4 * d, d), "muon"), ((d,), "adam")]
        out += [((d,), "adam"), ((d,), "adam")]
    elif kind == "llama":
        d, kv, ffn = case["d"], case["kv"], case["ffn"]
        out = [((case["vocab"], d), "adam")]
        for _ in range(case["layers"]):
            out += [((d,), "adam"), ((d, d), "muon"), ((kv, d), "muon"), ((kv, d), "muon"), ((d, d), "muon"),
                    ((d,), "adam"), ((ffn, d), "muon"), ((ffn, d), "muon"), ((d, ffn), "muon")]
        out += [((d,), "adam"), ((case["vocab"], d), "adam")]
    elif kind == "muon":
        out = [((case["rows"], case["cols"]), "muon")] * case["count"]
    elif kind == "adamw":
        out = [((n,), "adam") for n in _adamw_sizes(case)]
    return out


def _adamw_sizes(case):
    """Sizes spread evenly over their logarithm, in an order that mixes large and small; scaled to `total` if given."""
    n, lo, hi = case["tensors"], case["smallest"], case["largest"]
    if n == 1:
        return [hi]
    raw = [math.exp(math.log(lo) + (math.log(hi) - math.log(lo)) * ((i * 97) % n) / (n - 1)) for i in range(n)]
    scale = case["total"] / sum(raw) if case["total"] else 1.0
    return [max(1, min(hi, int(r * scale))) for r in raw]


def _flat(layout, packed):
    """(offset of each tensor, elements of the flat buffer); tensors start on 128-element boundaries unless packed."""
    offsets, at = [], 0
    for shape, _ in layout:
        offsets.append(at)
        n = math.prod(shape)
        at += n if packed else (n + 127) // 128 * 128
    return offsets, at


def _views(flat, layout, offsets):
    return [flat[o:o + math.prod(s)].view(s) for (s, _), o in zip(layout, offsets)]


def _normal(n, std, gen, dtype=torch.float32):
    return torch.empty(n, device="cuda").normal_(0.0, std, generator=gen).to(dtype)


def _part(layout, branch):
    return [e for e in layout if e[1] == branch]


def _step_inputs(case, seed):
    """Flat buffers of a step, per branch: parameters, gradients and the branch's state."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    layout = _layout(case)
    got = {}
    for branch in ("adam", "muon"):
        part = _part(layout, branch)
        if not part:
            continue
        offsets, n = _flat(part, case.get("packed", False))
        b = {"layout": part, "offsets": offsets, "param": _normal(n, 0.02, gen, dtype),
             "grad": _normal(n, 1e-3, gen, dtype)}
        if branch == "muon":
            b["momentum"] = _normal(n, 1e-3, gen)
        else:
            b["exp_avg"] = _normal(n, 1e-4, gen)
            b["exp_avg_sq"] = _normal(n, 1e-6, gen).abs_()
        got[branch] = b
    return got


def _matrix_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    r, c = case["rows"], case["cols"]
    if case["kind"] == "muon_step":
        return tuple(_normal(r * c, std, gen).view(r, c) for std in (0.02, 1e-3, 1e-3))
    # an iterate some way into the iteration: its largest singular value is about 1
    return _normal(r * c, 1.0 / (math.sqrt(r) + math.sqrt(c)), gen, torch.bfloat16).view(r, c)


# ---------------------------------------------------------------------------

def prepare(case, seed):
    from triton_muon_adamw import AdamConfig, MuonAdamW, MuonConfig
    from triton_muon_adamw.adamw import HipAdamW
    from triton_muon_adamw.muon import HipMuon

    kind = case["kind"]
    if kind == "muon_step":
        w, g, m = _matrix_inputs(case, seed)
        return {"kind": kind, "w": w, "g": g, "m": m, "out": torch.empty_like(w)}
    if kind == "ns_step":
        x = _matrix_inputs(case, seed)
        return {"kind": kind, "x": x, "out": torch.empty_like(x)}
    if kind == "ns_gram":
        x = _matrix_inputs(case, seed)
        return {"kind": kind, "x": x, "out": torch.empty((x.shape[0], x.shape[0]), dtype=x.dtype, device=x.device)}

    flat = _step_inputs(case, seed)
    params = {"adam": [], "muon": []}
    for branch, b in flat.items():
        for p, g in zip(_views(b["param"], b["layout"], b["offsets"]), _views(b["grad"], b["layout"], b["offsets"])):
            p = nn.Parameter(p)
            p.grad = g
            params[branch].append(p)
    if kind == "muon":
        opt = muon = HipMuon(params["muon"], **MUON)
        adamw = None
    elif kind == "adamw":
        opt = adamw = HipAdamW(params["adam"], **ADAM)
        muon = None
    else:
        opt = MuonAdamW(params, muon_config=MuonConfig(**MUON), adam_config=AdamConfig(**ADAM),
                        parameter_split="explicit")
        muon, adamw = opt.muon, opt.adamw
    if muon is not None:
        b = flat["muon"]
        for p, v in zip(params["muon"], _views(b["momentum"], b["layout"], b["offsets"])):
            muon.momentum[p] = v
    if adamw is not None:
        b = flat["adam"]
        for state, name in ((adamw.m, "exp_avg"), (adamw.v, "exp_avg_sq")):
            for p, v in zip(params["adam"], _views(b[name], b["layout"], b["offsets"])):
                state[p] = v
        adamw.step_num = PRIOR_STEPS
    scaler = None
    if case.get("amp"):
        # A scale of 1 that does not grow: the step is that of the gradients as they stand.
        scaler = torch.amp.GradScaler("cuda", init_scale=1.0, growth_interval=1 << 30)
        scaler.scale(torch.zeros((), device="cuda"))
    return {"kind": kind, "opt": opt, "scaler": scaler,
            "out": {branch: {k: b[k] for k in b if k not in ("layout", "offsets", "grad")} for branch, b in flat.items()}}


def run(state):
    from triton_muon_adamw.muon import muon_step, newton_shultz_step, solve_ns_kernel_1

    kind = state["kind"]
    if kind == "muon_step":
        rows, cols = state["w"].shape
        a, b, c = COEFFS
        muon_step(state["w"], state["g"], state["m"], MUON["beta"], a, b, c, MUON["lr"],
                  MUON["lr"] * math.sqrt(max(1, rows / cols)), MUON["weight_decay"], MUON["ns_steps"], MUON["eps"],
                  MUON["nesterov"], out=state["out"])
        return {"weights": state["w"], "momentum": state["m"], "update": state["out"]}
    if kind == "ns_step":
        newton_shultz_step(state["x"], *COEFFS, state["out"])
        return state["out"]
    if kind == "ns_gram":
        solve_ns_kernel_1(state["x"], state["out"])
        return state["out"]
    if state["scaler"] is not None:
        state["scaler"].step(state["opt"])
        state["scaler"].update()
    else:
        state["opt"].step()
    return state["out"]


def work(case):
    kind = case["kind"]
    if kind in ("muon_step", "ns_step", "ns_gram"):
        r, c = case["rows"], case["cols"]
        if kind == "ns_gram":  # the symmetric half of X X^T; read X, write the Gram
            return {"bytes": 2.0 * (r * c + r * r), "flops": float(r) * r * c}
        if kind == "ns_step":  # on the rows x cols matrix as it stands; read X, write the iterate
            return {"bytes": 4.0 * r * c, "flops": 3.0 * r * r * c + float(r) ** 3}
        m, n = min(r, c), max(r, c)  # read w, g, momentum; write w, momentum, update
        return {"bytes": 24.0 * r * c, "flops": MUON["ns_steps"] * (3.0 * m * m * n + float(m) ** 3)}
    half = 2 if case["dtype"] == "bf16" else 4
    nbytes = flops = 0.0
    for shape, branch in _layout(case):
        n = math.prod(shape)
        if branch == "adam":  # read p, g, m, v; write p, m, v
            nbytes += n * (3 * half + 16)
            flops += n * 14.0
        else:  # read p, g, momentum; write p, momentum
            nbytes += n * (3 * half + 8)
            lo, hi = min(shape), max(shape)
            flops += MUON["ns_steps"] * (3.0 * lo * lo * hi + float(lo) ** 3)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what torch's own arithmetic (bf16 Newton-Schulz with its sums in another order, fused AdamW)
    measured against this framework's: an orthogonalised update differs by 0.2-0.5% of its norm, of which a step of
    lr 0.02 leaves 0.3%/sqrt(cols) in parameters of std 0.02; bf16 parameters differ by the last place of the few
    whose rounding that turns; AdamW by fp32 rounding."""
    kind = case["kind"]
    if kind == "muon_step":
        return {"rel": 1.2e-2, "max": 0.1}
    if kind == "ns_step":
        return {"rel": 2e-3, "max": 0.03}
    if kind == "ns_gram":
        return {"rel": 5e-4, "max": 0.016}
    half = case["dtype"] == "bf16"
    if kind == "adamw":
        return {"rel": 4e-5, "max": 0.016} if half else {"rel": 1e-6, "max": 4e-6}
    cols = math.sqrt(min(s[1] for s, branch in _layout(case) if branch == "muon"))
    return {"rel": 0.012 / cols + (1e-3 if half else 0.0), "max": 0.6 / cols + (0.02 if half else 0.0)}


# ---------------------------------------------------------------------------
# float64, plain torch.

def _newton_schulz64(u, steps):
    a, b, c = COEFFS
    x = u.mT if u.shape[0] > u.shape[1] else u
    x = x / x.norm().clamp(min=MUON["eps"])
    for _ in range(steps):
        g = x @ x.mT
        x = a * x + (b * g + c * (g @ g)) @ x
    return x.mT if u.shape[0] > u.shape[1] else x


def _muon64(p, g, m):
    """(parameter, momentum, update) after one step, float64."""
    p, g, m = p.double(), g.double(), m.double()
    beta = MUON["beta"]
    m = m + (1 - beta) * (g - m)
    u = _newton_schulz64(g + beta * (m - g), MUON["ns_steps"])
    slr = MUON["lr"] * math.sqrt(max(1, p.shape[0] / p.shape[1]))
    return p * (1 - MUON["lr"] * MUON["weight_decay"]) - slr * u, m, u


def exact(case, seed):
    kind = case["kind"]
    if kind == "muon_step":
        w, m, u = _muon64(*_matrix_inputs(case, seed))
        return {"weights": w, "momentum": m, "update": u}
    if kind == "ns_step":
        x = _matrix_inputs(case, seed).double()
        a, b, c = COEFFS
        g = x @ x.mT
        return a * x + (b * g + c * (g @ g)) @ x
    if kind == "ns_gram":
        x = _matrix_inputs(case, seed).double()
        return x @ x.mT
    out = {}
    for branch, b in _step_inputs(case, seed).items():
        if branch == "muon":
            p64, m64 = b["param"].double(), b["momentum"].double()
            for p, g, m, po, mo in zip(*(_views(t, b["layout"], b["offsets"])
                                         for t in (b["param"], b["grad"], b["momentum"], p64, m64))):
                pn, mn, _ = _muon64(p, g, m)
                po.copy_(pn)
                mo.copy_(mn)
            # the gaps between tensors hold what they held
            out[branch] = {"param": p64, "momentum": m64}
        else:
            b1, b2 = ADAM["betas"]
            step = PRIOR_STEPS + 1
            keep = torch.zeros(b["param"].numel(), dtype=torch.bool, device="cuda")
            for (s, _), o in zip(b["layout"], b["offsets"]):
                keep[o:o + math.prod(s)] = True
            p, m, v = b["param"].double(), b["exp_avg"].double(), b["exp_avg_sq"].double()
            g = b["grad"].double()
            mn = b1 * m + (1 - b1) * g
            vn = b2 * v + (1 - b2) * g * g
            del g
            denom = (vn / (1 - b2**step)).sqrt() + ADAM["eps"]
            pn = p * (1 - ADAM["lr"] * ADAM["weight_decay"]) - ADAM["lr"] * (mn / (1 - b1**step)) / denom
            del denom
            out[branch] = {"param": torch.where(keep, pn, p), "exp_avg": torch.where(keep, mn, m),
                           "exp_avg_sq": torch.where(keep, vn, v)}
    return out
