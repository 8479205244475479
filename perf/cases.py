"""The work a user of this package has it do, as cases that can be timed and compared.

Four kinds of case, each one pass through public entry points:

  step      the two library calls that replace a wrapped projection's saved input and its weight
            gradient: `kernels.save_with_census` in the forward (coefficients, exact top-k residual,
            quantization) and `kernels.weight_grad` in the backward.  The same work bench.py reports
            as tokens/s.  Returns the coefficients, the quantization scale and dW; the residual
            entries are what the two calls hand to each other and reach the caller through dW.
  layer     one training step of the drop-in `STACRLinear`: Oja step and QR of the basis, dense
            forward, save, and the three gradients.
  adaptive  one training step of the adaptive engine's layer (energies, int8 coefficients, rank and
            refresh policy), as `apply_adaptive_stacr` installs it.
  hooks     the saved-tensor compressor: pack in the forward, unpack to the dense tensor in the
            backward.

Activations follow the generator of the configured workloads: rank-8 structure plus noise, 0.1 % of
the entries scaled by 20, optionally a log-normal scale per channel; gradients are normal.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "stac-r_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "stac-r_amd"))

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}
CHUNK_ROWS = 512
OJA_LR = 0.01  # STACRLinear's and the compressor's default


def _step(name, rows, d_in, d_out, rank=8, dtype="bf16", mode="chunk_topk", budget=0.005, bits=8, conv1d=False,
          lognormal=False):
    case = {"kind": "step", "rows": rows, "d_in": d_in, "d_out": d_out, "rank": rank, "dtype": dtype, "mode": mode,
            "budget": budget, "bits": bits, "conv1d": conv1d, "lognormal": lognormal}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one short sequence through a square projection: launches and host time are all there is
        _step("step_small", 512, 768, 768),
        # GPT-2-medium MLP c_fc at batch 8 x 1024, the headline layer, and its c_proj
        _step("step_c_fc", 8192, 1024, 4096, mode="global_topk", conv1d=True, lognormal=True),
        _step("step_c_proj", 8192, 4096, 1024, mode="global_topk", conv1d=True, lognormal=True),
        # fp32 training of a 768 -> 3072 MLP layer
        _step("step_fp32", 4096, 768, 3072, dtype="f32"),
        # Turbo: frozen basis, no residual
        _step("step_turbo", 8192, 1280, 5120, budget=0.0, conv1d=True),
        # the 2048 <-> 8192 MLP of a 1.4 B model at 16 x 2048 tokens, rank 16
        _step("step_wide_up", 32768, 2048, 8192, rank=16),
        _step("step_wide_down", 32768, 8192, 2048, rank=16),
        # a ragged last batch in fp16 with 4-bit residuals; features that no tile divides
        _step("step_ragged", 3001, 1000, 3000, dtype="f16", budget=0.01, bits=4),
        # the drop-in layer as apply_stacr leaves it (chunk top-k, basis refreshed every step)
        {"name": "layer_step", "kind": "layer", "rows": 8192, "d_in": 1024, "d_out": 4096, "rank": 8},
        # the adaptive engine's layer: int8 coefficients, sensitivity rank control, hybrid refresh
        {"name": "adaptive_step", "kind": "adaptive", "rows": 8192, "d_in": 2048, "d_out": 8192, "rank": 16},
        # the saved-tensor hooks on a GPT-2-medium activation
        {"name": "hooks_pack_unpack", "kind": "hooks", "rows": 8192, "d_in": 1024, "rank": 8, "dtype": "bf16"},
    ]


# a drawn case moves at most what the largest listed step does; the forms that are rarely trained at
# that size (fp16 and fp32, whole layers, features off the multiples of 64) at most what c_fc's does
_MOST = 32768 * (2048 + 8192)
_MOST_OTHER = 8192 * (1024 + 4096)


def _log_between(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _features(rng):
    d = int(_log_between(rng, 256, 8192))
    u = rng.random()
    if u < 0.7:
        return max(256, d // 64 * 64)
    return d // 8 * 8 if u < 0.9 else d | 1


def draw(rng):
    kind = rng.choice(["step"] * 7 + ["layer", "adaptive", "hooks"])
    rows = int(_log_between(rng, 256, 32768))
    if rng.random() < 0.6:
        rows = rows // 128 * 128
    d_in, d_out = _features(rng), _features(rng)
    rank = rng.choice([4, 8, 8, 8, 16])
    if kind == "step":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        plain = dtype == "bf16" and d_in % 64 == 0 and d_out % 64 == 0
        rows = max(64, min(rows, (_MOST if plain else _MOST_OTHER) // (d_in + d_out)))
        return _step(None, rows, d_in, d_out, rank=rank, dtype=dtype, mode=rng.choice(["chunk_topk", "global_topk"]),
                     budget=rng.choice([0.005, 0.005, 0.005, 0.01, 0.002, 0.0]), bits=rng.choice([8, 8, 8, 4, 0]),
                     conv1d=rng.random() < 0.5, lognormal=rng.random() < 0.5)
    d_in, d_out = max(256, d_in // 64 * 64), max(256, d_out // 64 * 64)
    rows = max(64, min(rows, _MOST_OTHER // (d_in + d_out)))
    if kind == "hooks":
        return {"kind": kind, "rows": rows, "d_in": d_in, "rank": rank, "dtype": rng.choice(["bf16", "f16"])}
    return {"kind": kind, "rows": rows, "d_in": d_in, "d_out": d_out, "rank": rank}


# ------------------------------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _activation(gen, rows, d, dtype, lognormal=False, structure=None):
    dev = gen.device
    b = torch.randn(d, 8, generator=gen, device=dev) if structure is None else structure
    x = torch.randn(rows, 8, generator=gen, device=dev) @ b.t()
    x += 0.05 * torch.randn(rows, d, generator=gen, device=dev)
    x = torch.where(torch.rand(rows, d, generator=gen, device=dev) < 0.001, x * 20.0, x)
    if lognormal:
        x *= torch.exp(torch.randn(d, generator=gen, device=dev))
    return x.to(dtype)


def _orthonormal(gen, d, rank):
    return torch.linalg.qr(torch.randn(d, rank, generator=gen, device=gen.device).cpu())[0].to(gen.device).contiguous()


def _inputs(case, seed):
    """The tensors a case starts from, from its seed alone."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    kind, rows, d_in, rank = case["kind"], case["rows"], case["d_in"], case["rank"]
    dtype = DTYPES[case.get("dtype", "bf16")]
    if kind == "hooks":
        b = torch.randn(d_in, 8, generator=gen, device=dev)
        return {"first": _activation(gen, 64, d_in, dtype, structure=b),
                "x": _activation(gen, rows, d_in, dtype, structure=b)}
    x = _activation(gen, rows, d_in, dtype, case.get("lognormal", False))
    q = _orthonormal(gen, d_in, rank)
    g = torch.randn(rows, case["d_out"], generator=gen, device=dev).to(dtype)
    if kind == "step":
        return {"x": x, "q": q.to(dtype), "g": g}
    w = (torch.randn(case["d_out"], d_in, generator=gen, device=dev) * d_in**-0.5).to(dtype)
    b = (torch.randn(case["d_out"], generator=gen, device=dev) * 0.02).to(dtype)
    return {"x": x, "q": q, "g": g, "w": w, "b": b}


def _linear(s):
    lin = torch.nn.Linear(s["w"].shape[1], s["w"].shape[0], device=s["w"].device, dtype=s["w"].dtype)
    with torch.no_grad():
        lin.weight.copy_(s["w"])
        lin.bias.copy_(s["b"])
    return lin


def prepare(case, seed):
    """What the program holds before the pass: the inputs, and the layer or compressor it keeps
    from step to step (resumed from a basis, as from a checkpoint)."""
    s = {"case": case, **_inputs(case, seed)}
    if case["kind"] == "layer":
        from stacr_amd import STACRLinear

        layer = STACRLinear.from_linear(_linear(s), rank=case["rank"]).train()
        layer.load_state_dict({"basis": s["q"], "basis_ready": torch.tensor(True), "_last_update_step": torch.tensor(0)},
                              strict=False)
        s.update(layer=layer, step=0)
        s["x"].requires_grad_(True)
    elif case["kind"] == "adaptive":
        from stacr_amd import AdaptiveSTACRConfig, apply_adaptive_stacr

        cfg = AdaptiveSTACRConfig(rank=case["rank"], rank_mode="sensitivity", rank_min=4, rank_max=case["rank"],
                                  rank_adjust_interval=5, residual_mode="topk", residual_budget=0.005,
                                  quantize_coefficients=True, quantize_residuals=True, residual_quantize_bits=8,
                                  refresh_trigger="hybrid", refresh_period=10, refresh_energy_threshold=0.1,
                                  basis_dtype="bfloat16")
        model = torch.nn.Sequential(_linear(s)).train()
        layer = apply_adaptive_stacr(model, cfg, surface="all", min_features=1)[0]
        layer.load_state_dict({"basis": s["q"], "_basis_initialized": torch.tensor([True])}, strict=False)
        s.update(model=model, layer=layer, step=0)
        s["x"].requires_grad_(True)
    elif case["kind"] == "hooks":
        from stacr_amd import STACRCompressor, STACRConfig

        s["compressor"] = STACRCompressor(STACRConfig(rank=case["rank"], min_numel=1))
        s["compressor"].pack(s["first"])  # the basis is fitted to the first activation it sees
    return s


# --------------------------------------------------------------------------------------- passes
def _run_step(s):
    from stacr_amd import kernels

    c = s["case"]
    coeff, idx, data, scale, census = kernels.save_with_census(s["x"], s["q"], mode=c["mode"], budget=c["budget"],
                                                               chunk_rows=CHUNK_ROWS, bits=c["bits"])
    residual = (idx, data, scale) if idx is not None else None
    dw, _ = kernels.weight_grad(s["g"], coeff, s["q"], residual, c["bits"], c["conv1d"], s["x"].dtype, census=census)
    return {"coeff": coeff, "dw": dw, "scale": scale}


def _run_layer(s):
    layer = s["layer"]
    s["step"] += 1
    layer.set_step(s["step"])
    s["x"].grad = layer.weight.grad = layer.bias.grad = None
    y = layer(s["x"])
    y.backward(s["g"])
    return {"y": y.detach(), "dx": s["x"].grad, "dw": layer.weight.grad, "db": layer.bias.grad, "basis": layer.basis}


def _run_adaptive(s):
    from stacr_amd import set_stacr_runtime_state

    layer = s["layer"]
    s["step"] += 1
    set_stacr_runtime_state(s["model"], s["step"])
    s["x"].grad = layer.linear.weight.grad = layer.linear.bias.grad = None
    y = s["model"](s["x"])
    y.backward(s["g"])
    return {"y": y.detach(), "dx": s["x"].grad, "dw": layer.linear.weight.grad, "db": layer.linear.bias.grad,
            "basis": layer.effective_basis}


def _run_hooks(s):
    packed = s["compressor"].pack(s["x"])
    return {"dense": s["compressor"].unpack(packed), "coeff": packed.coeff}


def run(state):
    return {"step": _run_step, "layer": _run_layer, "adaptive": _run_adaptive,
            "hooks": _run_hooks}[state["case"]["kind"]](state)


# ---------------------------------------------------------------------------- what a pass needs
def _entries(case):
    return round(case.get("budget", 0.005) * case["rows"] * case["d_in"])


def work(case):
    """Each input read once, each output written once; entries as int32 index plus stored value."""
    n, d_in, rank, k = case["rows"], case["d_in"], case["rank"], _entries(case)
    size = SIZE[case.get("dtype", "bf16")]
    project = 2 * n * d_in * rank
    if case["kind"] == "hooks":  # Oja step, projection, residual; X in, C and the entries, dense X out
        return {"bytes": 2 * n * d_in * size + n * rank * size + k * (8 + size) + 2 * 4 * d_in * rank,
                "flops": 5 * project}
    d_out = case["d_out"]
    entry = 4 + {8: 1, 4: 0.5, 0: size}[case.get("bits", 8)] if k else 0
    save = n * d_in * size + 4 * d_in * rank + n * rank * size + k * entry
    grad = n * d_out * size + n * rank * size + k * entry + 4 * d_in * rank + d_in * d_out * size
    flops = 2 * project + 2 * n * d_out * rank + 2 * d_in * d_out * rank + 2 * k * d_out
    if case["kind"] != "step":  # Y and dX: the weight twice, X again, Y out, dX out
        save += d_in * d_out * size + n * d_out * size
        grad += d_in * d_out * size + n * d_in * size + d_out * size
        flops += 2 * 2 * n * d_in * d_out + 2 * project
    return {"bytes": save + grad, "flops": flops}


def tolerance(case):
    """About four times what one rounding of the outputs shows against `exact` (bf16 1.7e-3, fp16
    2.1e-4); fp32 sums are within 2e-7 of it.  "max" leaves room for a residual code or entry that
    another order of the 16-bit coefficients' sums moves."""
    dtype = case.get("dtype", "bf16")
    if dtype == "f32":
        return {"rel": 1e-5}
    return {"rel": 8e-3 if dtype == "bf16" else 1e-3, "max": 0.1}


# ------------------------------------------------------------------- the same outputs in 64 bits
def _top(r, k):
    """Flat positions of the k largest |r|, ties to the lowest position, ascending."""
    mag = r.abs()
    cut = torch.topk(mag, k).values.min()
    above = (mag > cut).nonzero().flatten()
    tie = (mag == cut).nonzero().flatten()[: k - above.numel()]
    return torch.cat((above, tie)).sort().values


def _select(r, case):
    total = r.numel()
    k_total = round(case.get("budget", 0.005) * total)
    if k_total <= 0:
        return None
    flat = r.reshape(-1)
    if case.get("mode", "chunk_topk") == "global_topk":
        return _top(flat, k_total)
    size, parts = CHUNK_ROWS * r.shape[1], []
    for start in range(0, total, size):
        part = flat[start:start + size]
        parts.append(_top(part, max(1, min(part.numel(), round(case.get("budget", 0.005) * part.numel())))) + start)
    pos = torch.cat(parts)
    return pos if pos.numel() <= k_total else pos[_top(flat[pos], k_total)]


def _factors(x, q, case):
    """(coefficients in 64 bits, the activation its saved factors stand for, the scale): what is
    stored is rounded to its stored type, everything between is in 64 bits."""
    dtype, bits = x.dtype, case.get("bits", 8)
    coeff = x.double() @ q.double()
    approx = coeff.to(dtype).double() @ q.double().t()
    r = (x.double() - approx.to(dtype).double()).to(dtype).double()
    pos, scale = _select(r, case), None
    if pos is not None:
        v, scale = r.reshape(-1)[pos], 1.0
        if bits:
            qmax = 127 if bits == 8 else 7
            s = (v.abs().max() / qmax).clamp_min(torch.finfo(torch.float32).tiny).float().double()
            v, scale = torch.round(v / s).clamp(-qmax - 1, qmax) * s, float(s)
        approx.view(-1)[pos] += v
    return coeff, approx, scale


def _oja(x, q):
    """One Oja step in 64 bits, then the reduced QR (LAPACK's signs)."""
    x, q = x.double(), q.double()
    y = x @ q
    stepped = q + OJA_LR * (x.t() @ y - q @ (y.t() @ y)) / x.shape[0]
    return torch.linalg.qr(stepped.cpu())[0].to(x.device)


def exact(case, seed):
    s = _inputs(case, seed)
    x, kind = s["x"], case["kind"]
    if kind == "hooks":
        start = torch.linalg.svd(s["first"].double().cpu(), full_matrices=False)[2][: case["rank"]].t().to(x.device)
        q = _oja(x, start).to(x.dtype)  # C depends on the vectors' signs, the dense tensor does not
        return {"dense": _factors(x, q, {**case, "mode": "global_topk", "bits": 0})[1], "coeff": None}
    g = s["g"].double()
    if kind == "step":
        coeff, approx, scale = _factors(x, s["q"], case)
        dw = g.t() @ approx
        return {"coeff": coeff, "dw": dw.t() if case["conv1d"] else dw, "scale": scale}
    w, b = s["w"].double(), s["b"].double()
    out = {"y": x.double() @ w.t() + b, "dx": g @ w, "db": g.sum(0), "dw": None, "basis": None}
    if kind == "layer":  # the adaptive engine's gradient and basis follow its own rank and refresh policy
        out["basis"] = _oja(x, s["q"])
        out["dw"] = g.t() @ _factors(x, out["basis"].float().to(x.dtype), case)[1]
    return out
