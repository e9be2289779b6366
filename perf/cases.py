"""Performance cases of the BF16 training path, through the package's public entry points.

``listed()`` names the cases, ``draw(rng)`` gives another of the same ranges. A case is a
dict with a ``kind`` and its sizes:

* ``rmsnorm``: the RMSNorm operator on a BF16 residual stream, forward and backward.
* ``swiglu``: the standalone SwiGLU operator on a packed projection, forward and backward.
* ``layout``: the packed attention-backward gradient, one launch of a prepared callable.
* ``swiglu_mm``: the paired up/gate projection with the SwiGLU epilogue, forward.
* ``projection``: RMSNorm, input projection and gate sigmoid, forward.
* ``projection_grad``: the backward of ``projection`` into a cleared FP32 gradient buffer.
* ``linear``: a projection's three products on the GEMM kernels: Y, dX and the BF16 dW.
* ``ffn``: norm2 and the SwiGLU block of a core with its residual add, forward and
  backward from FP32 master weights, as the training adapter runs them.
* ``head``: the tied LM head's cross-entropy with the gradients of the hidden state and of
  the FP32 head weight.

Model widths run from 512 to 2048 (the default configuration's 1280, the layer
benchmark's 2048), tokens per call from 128 (one chunk of the default configuration) to
16384 (the layer benchmark), vocabularies up to 32768.
"""

from __future__ import annotations

import os
import sys

import torch

_package = os.path.abspath("warpstate-ai_amd")
if _package not in sys.path:
    sys.path.insert(0, _package)

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
EPS = 1e-5
IGNORED = -100
# A tile request the training adapter makes for its paired projection.
SWIGLU_TILE = (128, 128, 32, 8, 3)


def listed():
    return [
        # The smallest call: the norm of four 128-token chunks at the default width, where
        # launches and the operator's own overhead are what a training step waits for.
        {"name": "rmsnorm_512x1280", "kind": "rmsnorm", "rows": 512, "d": 1280, "eager": True},
        # Standalone SwiGLU at the reference's production shape (8192 tokens, ffn 7168).
        {"name": "swiglu_8192x7168", "kind": "swiglu", "rows": 8192, "h": 7168, "eager": False},
        # The packed attention-backward gradient at the profiled shape.
        {"name": "layout_profile", "kind": "layout", "b": 4, "n": 16, "h": 32, "c": 128, "hd": 64},
        # The FFN half of a default-configuration core on four chunks: a small batch.
        {"name": "ffn_512", "kind": "ffn", "rows": 512, "d": 1280, "ffn": 4480},
        # The same core on a ragged last batch of an epoch.
        {"name": "ffn_ragged_1999", "kind": "ffn", "rows": 1999, "d": 1280, "ffn": 4480},
        # The FFN half of the benchmarked layer, forward and backward: the bulk of a step.
        {"name": "ffn_16384", "kind": "ffn", "rows": 16384, "d": 2048, "ffn": 5632},
        # The paired SwiGLU projection of a 1024-wide model (first benchmark configuration).
        {"name": "swiglu_mm_4096", "kind": "swiglu_mm", "rows": 4096, "d": 1024, "h": 2816,
         "algorithm": "tiled", "eager": True},
        # The benchmarked layer's input projection with its norm and gate sigmoid.
        {"name": "projection_16384", "kind": "projection", "rows": 16384, "d": 2048, "n": 9216,
         "gate_begin": 6144, "gate_end": 8192},
        # The input projection's backward in a default-configuration core, 32 chunks,
        # into the FP32 gradient buffer that the optimizer keeps.
        {"name": "projection_grad_4096", "kind": "projection_grad", "rows": 4096, "d": 1280,
         "n": 6400, "gate_begin": 3840, "gate_end": 5120},
        # The three products of the reference's measured input projection, BF16 throughout.
        {"name": "linear_8192", "kind": "linear", "rows": 8192, "d": 2048, "n": 10240,
         "algorithm": "persistent"},
        # The head of a small batch whose rows are no multiple of a tile.
        {"name": "head_1000", "kind": "head", "rows": 1000, "d": 1280, "vocab": 32768},
        # The head of the benchmarked batch: the largest call.
        {"name": "head_16384", "kind": "head", "rows": 16384, "d": 2048, "vocab": 32768},
    ]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def _rows(rng):
    """Tokens of a call: whole 128-token chunks, or any count (a ragged or packed batch)."""
    rows = _log(rng, 128, 16384)
    return max(128, rows // 128 * 128) if rng.random() < 0.5 else rows


def _width(rng, low=512, high=2048):
    """A feature width: a multiple of 64, now and then of 8 only."""
    step = 8 if rng.random() < 0.2 else 64
    return _log(rng, low, high) // step * step


def draw(rng):
    kind = rng.choice(["rmsnorm", "swiglu", "layout", "swiglu_mm", "projection",
                       "projection_grad", "linear", "ffn", "head"])
    case = {"kind": kind}
    if kind == "layout":
        case.update(b=rng.randint(1, 4), n=_log(rng, 1, 16), h=rng.choice([8, 16, 20, 32]),
                    c=rng.choice([32, 64, 100, 128]), hd=rng.choice([64, 128]))
        return case
    case["rows"] = _rows(rng)
    if kind in ("rmsnorm", "swiglu", "swiglu_mm"):
        case["eager"] = rng.random() < 0.5
    if kind == "swiglu":
        case["h"] = _width(rng, 1024, 7168)
        return case
    case["d"] = _width(rng)
    if kind == "swiglu_mm":
        case.update(h=_width(rng, 1024, 7168), algorithm=rng.choice(["tiled", "persistent"]))
    elif kind in ("projection", "projection_grad"):
        case.update(n=5 * case["d"], gate_begin=3 * case["d"], gate_end=4 * case["d"])
    elif kind == "linear":
        case.update(n=_width(rng, 512, 10240), algorithm=rng.choice(["tiled", "persistent"]))
    elif kind == "ffn":
        case["ffn"] = _width(rng, 1024, 7168)
    elif kind == "head":
        # Trained vocabularies are padded to a multiple of 128; some are not.
        vocab = _log(rng, 4096, 32768)
        case["vocab"] = vocab // 128 * 128 if rng.random() < 0.7 else vocab
    return case


# --- inputs --------------------------------------------------------------------------------

class _Draw:
    """Normal draws on the GPU from one seeded generator, FP32 rounded to the wanted type."""

    def __init__(self, seed):
        self.gen = torch.Generator("cuda").manual_seed(seed)

    def __call__(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        t = torch.randn(shape, generator=self.gen, device="cuda", dtype=F32)
        return t.mul_(std).add_(mean).to(dtype)


def _inputs(case, seed):
    """The tensors of a case in the distributions a step sees: unit-variance activations,
    N(0, 0.02) weights, gradients of 1e-2, norm weights near 1."""
    kind, draws = case["kind"], _Draw(seed)
    if kind == "layout":
        from ops.backward_layout import make_inputs

        shape = (case["b"], case["n"], case["h"], case["c"], case["hd"])
        return {"inputs": make_inputs(shape, device="cuda", seed=seed)}
    rows = case["rows"]
    if kind == "swiglu":
        return {"packed": draws(rows, 2 * case["h"]), "grad": draws(rows, case["h"], std=1e-2)}
    d = case["d"]
    if kind == "swiglu_mm":
        return {"x": draws(rows, d), "weight": draws(2 * case["h"], d, std=0.02)}
    if kind == "linear":
        return {"x": draws(rows, d), "weight": draws(case["n"], d, std=0.02),
                "grad": draws(rows, case["n"], std=1e-2)}
    if kind == "head":
        targets = torch.randint(0, case["vocab"], (rows,), generator=draws.gen, device="cuda")
        ignored = torch.rand((rows,), generator=draws.gen, device="cuda") < 0.05
        return {"hidden": draws(rows, d), "weight": draws(case["vocab"], d, std=0.02, dtype=F32),
                "targets": targets.masked_fill_(ignored, IGNORED)}
    t = {"x": draws(rows, d), "norm": draws(d, std=0.1, mean=1.0, dtype=F32)}
    if kind == "rmsnorm":
        t["grad"] = draws(rows, d, std=1e-2)
    elif kind in ("projection", "projection_grad"):
        t["weight"] = draws(case["n"], d, std=0.02)
        if kind == "projection_grad":
            t["grad"] = draws(rows, case["n"], std=1e-2)
    elif kind == "ffn":
        t.update(w_upgate=draws(2 * case["ffn"], d, std=0.02, dtype=F32),
                 w_down=draws(d, case["ffn"], std=0.02, dtype=F32),
                 grad=draws(rows, d, std=1e-2))
    return t


def prepare(case, seed):
    state = _inputs(case, seed)
    state["case"] = case
    kind = case["kind"]
    if kind == "layout":
        from ops.backward_layout import prepare_layout

        state["launch"] = prepare_layout(state["inputs"], "single")
    elif kind == "swiglu":
        state["packed"].requires_grad_(True)
    elif kind == "rmsnorm":
        state["x"].requires_grad_(True)
        state["norm"].requires_grad_(True)
    elif kind == "ffn":
        for name in ("x", "norm", "w_upgate", "w_down"):
            state[name].requires_grad_(True)
    elif kind == "head":
        state["hidden"].requires_grad_(True)
        state["weight"].requires_grad_(True)
    elif kind == "projection_grad":
        # What the forward saved, in its rounding: rstd, y = r(r(x rstd) r(w)) and the
        # projection with its gate columns through the sigmoid.
        x = state["x"].float()
        rstd = torch.rsqrt(x.square().mean(-1) + EPS)
        state["rstd"] = rstd
        state["normed"] = (x * rstd[:, None]).to(BF16) * state["norm"].to(BF16)
        out = state["normed"] @ state["weight"].T
        gate = slice(case["gate_begin"], case["gate_end"])
        out[:, gate] = torch.sigmoid(out[:, gate])
        state["out"] = out
        state["weight_grad"] = torch.zeros(state["weight"].shape, dtype=F32, device="cuda")
    return state


# --- one pass ------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "rmsnorm":
        from ops.activation_execution import bf16_rmsnorm

        y, _rstd = bf16_rmsnorm(state["x"], state["norm"], EPS, case["eager"])
        dx, dnorm = torch.autograd.grad(y, [state["x"], state["norm"]], state["grad"])
        return {"y": y, "dx": dx, "dnorm": dnorm}
    if kind == "swiglu":
        from ops.activation_execution import bf16_swiglu

        act = bf16_swiglu(state["packed"], case["eager"])
        dpacked, = torch.autograd.grad(act, [state["packed"]], state["grad"])
        return {"act": act, "dpacked": dpacked}
    if kind == "layout":
        return {"packed": state["launch"]()}
    if kind == "swiglu_mm":
        from ops.matmul_epilogue import launch_swiglu_mm

        packed, act = launch_swiglu_mm(state["x"], state["weight"].T, case["algorithm"],
                                       SWIGLU_TILE, case["eager"])
        return {"packed": packed, "act": act}
    if kind == "projection":
        from ops.fused_execution import rmsnorm_gate_mm

        out, rstd = rmsnorm_gate_mm(state["x"], state["norm"], EPS, state["weight"],
                                    (case["gate_begin"], case["gate_end"]))
        return {"out": out, "rstd": rstd}
    if kind == "projection_grad":
        from ops.fused_execution import rmsnorm_gate_mm_backward

        grad = state["weight_grad"].zero_()  # the optimizer's cleared gradient
        dx, dnorm = rmsnorm_gate_mm_backward(
            state["x"], state["norm"], state["rstd"], state["normed"], state["weight"],
            (case["gate_begin"], case["gate_end"]), state["out"], state["grad"], grad)
        return {"dx": dx, "dnorm": dnorm, "dweight": grad}
    if kind == "linear":
        from ops.matmul_kernels import launch_mm

        x, weight, grad, algorithm = state["x"], state["weight"], state["grad"], case["algorithm"]
        return {"y": launch_mm(x, weight.T, algorithm), "dx": launch_mm(grad, weight, algorithm),
                "dweight": launch_mm(grad.T, x, algorithm)}
    if kind == "ffn":
        from ops.activation_execution import bf16_rmsnorm
        from ops.fused_training import fused_swiglu_block

        x, norm, w_upgate, w_down = (state[k] for k in ("x", "norm", "w_upgate", "w_down"))
        h, _rstd = bf16_rmsnorm(x, norm, EPS, True)
        y = fused_swiglu_block(h, w_upgate, w_down, x)[0]
        dx, dnorm, dup, ddown = torch.autograd.grad(y, [x, norm, w_upgate, w_down], state["grad"])
        return {"y": y, "dx": dx, "dnorm": dnorm, "dw_upgate": dup, "dw_down": ddown}
    if kind == "head":
        from ops.fused_execution import linear_cross_entropy

        mean, loss = linear_cross_entropy(state["hidden"], state["weight"], state["targets"])
        dhidden, dweight = torch.autograd.grad(mean, [state["hidden"], state["weight"]])
        return {"mean": mean, "loss": loss, "dhidden": dhidden, "dweight": dweight}
    raise ValueError(f"unknown kind {kind!r}")


def work(case):
    kind = case["kind"]
    if kind == "layout":
        elements = case["b"] * case["n"] * case["h"] * case["c"] * case["hd"]
        tables = 2 * 4 * case["c"] * case["hd"]
        return {"bytes": 34 * elements + tables, "flops": 0}  # 12 inputs, 5 sections, BF16
    rows = case["rows"]
    if kind == "swiglu":
        # packed, grad in; act, dpacked out.
        return {"bytes": 2 * rows * case["h"] * (2 + 1 + 1 + 2), "flops": 0}
    d = case["d"]
    if kind == "rmsnorm":
        return {"bytes": 2 * rows * d * 4 + 4 * d * 2 + 4 * rows, "flops": 0}
    if kind == "swiglu_mm":
        h = case["h"]
        return {"bytes": 2 * (rows * d + 2 * h * d + 3 * rows * h), "flops": 4 * rows * d * h}
    if kind == "projection":
        n = case["n"]
        return {"bytes": 2 * (rows * d + n * d + rows * n) + 4 * (rows + d),
                "flops": 2 * rows * d * n}
    if kind == "projection_grad":
        n, gate = case["n"], case["gate_end"] - case["gate_begin"]
        inputs = 2 * (2 * rows * d + n * d + rows * n + rows * gate) + 4 * (rows + d)
        return {"bytes": inputs + 2 * rows * d + 4 * (d + n * d), "flops": 4 * rows * d * n}
    if kind == "linear":
        n = case["n"]
        return {"bytes": 4 * (rows * d + n * d + rows * n), "flops": 6 * rows * d * n}
    if kind == "ffn":
        weights = 3 * case["ffn"] * d
        return {"bytes": 2 * 4 * rows * d + 4 * 2 * (weights + d), "flops": 6 * rows * weights}
    vocab = case["vocab"]
    return {"bytes": 2 * 2 * rows * d + 4 * 2 * vocab * d + 12 * rows,
            "flops": 6 * rows * vocab * d}


def tolerance(case):
    """About four times the largest 2-norm error measured against the same sums in 64 bits:
    one BF16 rounding (1.7e-3) for single products and the layout, two to four in a chain for
    the rest (rmsnorm 2.9e-3, swiglu 2.4e-3, swiglu_mm 3.5e-3, projection 3.3e-3,
    projection_grad 3.4e-3, ffn 5.9e-3, head 3.9e-3)."""
    return {"rel": {"rmsnorm": 1.2e-2, "swiglu": 1e-2, "layout": 7e-3, "swiglu_mm": 1.4e-2,
                    "projection": 1.3e-2, "projection_grad": 1.4e-2, "linear": 7e-3,
                    "ffn": 2.4e-2, "head": 1.6e-2}[case["kind"]]}


# --- the same values in 64 bits -------------------------------------------------------------

def _rms(x, w):
    rstd = torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return x * rstd * w, rstd


def _swiglu(packed):
    up, gate = packed.chunk(2, dim=-1)
    return up * gate * torch.sigmoid(gate)


def _token_major(t):
    b, n, h, c, d = t.shape
    return t.transpose(2, 3).reshape(b, n * c, h * d)


def _exact_layout(inputs):
    f = {k: v.to(F64) for k, v in zip(inputs._fields, inputs)}
    b, n, h, c, d = f["q_memory"].shape

    def unrotate(t):
        pairs = t.unflatten(-1, (-1, 2))
        return torch.stack((pairs[..., 1], -pairs[..., 0]), dim=-1).flatten(-2)

    q = f["q_memory"] + f["q_local"]
    k = f["k_write"].transpose(-2, -1) * (1 - f["tanh_k"] ** 2) + f["k_local"]
    dy = f["grad_y"].view(b, n, c, h, d).transpose(2, 3)
    gate = f["gate"]
    sections = (unrotate(q * f["sin"]) + q * f["cos"], unrotate(k * f["sin"]) + k * f["cos"],
                f["v_local"], dy * (f["local"] - f["memory"] * d ** -0.5) * gate * (1 - gate),
                f["u_write"] * (1 - f["tanh_u"] ** 2))
    return torch.cat([_token_major(s) for s in sections], dim=-1)


def exact(case, seed):
    """The outputs of ``run`` in 64-bit arithmetic from the same inputs."""
    kind = case["kind"]
    t = _inputs(case, seed)
    if kind == "layout":
        return {"packed": _exact_layout(t["inputs"])}
    # Inputs that are BF16, and masters that the path rounds to BF16, are exact in 64 bits.
    master = {"w_upgate", "w_down"} | ({"weight"} if kind == "head" else set())
    f = {k: v if v.dtype == torch.int64 else (v.to(BF16) if k in master else v).to(F64)
         for k, v in t.items()}
    if kind == "rmsnorm":
        x, w = f["x"].requires_grad_(True), f["norm"].requires_grad_(True)
        y, _rstd = _rms(x, w)
        dx, dnorm = torch.autograd.grad(y, [x, w], f["grad"])
        return {"y": y.detach(), "dx": dx, "dnorm": dnorm}
    if kind == "swiglu":
        packed = f["packed"].requires_grad_(True)
        act = _swiglu(packed)
        dpacked, = torch.autograd.grad(act, [packed], f["grad"])
        return {"act": act.detach(), "dpacked": dpacked}
    if kind == "swiglu_mm":
        packed = f["x"] @ f["weight"].T
        return {"packed": packed, "act": _swiglu(packed)}
    if kind == "projection":
        y, rstd = _rms(f["x"], f["norm"])
        out = y @ f["weight"].T
        gate = slice(case["gate_begin"], case["gate_end"])
        out[:, gate] = torch.sigmoid(out[:, gate])
        return {"out": out, "rstd": rstd[:, 0]}
    if kind == "projection_grad":
        # From the tensors the forward saved, as the call takes them.
        s = prepare(case, seed)
        dp = f["grad"].clone()
        gate = slice(case["gate_begin"], case["gate_end"])
        saved = s["out"][:, gate].to(F64)
        dp[:, gate] *= (1 - saved) * saved
        dy = dp @ f["weight"]
        r = s["rstd"].to(F64)[:, None]
        dz = dy * f["norm"]
        dr = (dz * f["x"]).mean(-1, keepdim=True)
        return {"dx": dz * r - f["x"] * r ** 3 * dr, "dnorm": (dy * f["x"] * r).sum(0),
                "dweight": dp.T @ s["normed"].to(F64)}
    if kind == "linear":
        return {"y": f["x"] @ f["weight"].T, "dx": f["grad"] @ f["weight"],
                "dweight": f["grad"].T @ f["x"]}
    if kind == "ffn":
        leaves = [f[k].requires_grad_(True) for k in ("x", "norm", "w_upgate", "w_down")]
        x, norm, w_upgate, w_down = leaves
        y = x + _swiglu(_rms(x, norm)[0] @ w_upgate.T) @ w_down.T
        dx, dnorm, dup, ddown = torch.autograd.grad(y, leaves, f["grad"])
        return {"y": y.detach(), "dx": dx, "dnorm": dnorm, "dw_upgate": dup, "dw_down": ddown}
    targets, valid = f["targets"], f["targets"] != IGNORED
    count = valid.sum().clamp_min(1)
    index = targets.clamp_min(0)[:, None]
    logits = f["hidden"] @ f["weight"].T
    lse = torch.logsumexp(logits, -1)
    loss = (lse - logits.gather(1, index)[:, 0]) * valid
    grad = logits.sub_(lse[:, None]).exp_()
    grad.scatter_add_(1, index, -torch.ones_like(index, dtype=F64))
    grad *= (valid / count)[:, None]
    return {"mean": loss.sum() / count, "loss": loss, "dhidden": grad @ f["weight"],
            "dweight": grad.T @ f["hidden"]}
