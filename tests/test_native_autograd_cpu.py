"""The native autograd nodes under compiled autograd and torch.compile, on the CPU.

``csrc/autograd.cpp`` is compiled once more with its kernels registered for CPU tensors, and
loaded in a process of its own where the operators have plain PyTorch kernels. Every
operator's backward must then give the eager gradients when compiled autograd traces it
(which asks more of a C++ node than the engine does) and when the call is compiled.
"""
import json
import subprocess
import sys
from pathlib import Path

import pytest

import build_lib

ROOT = Path(__file__).resolve().parents[1]
NAMES = ["swiglu", "rmsnorm", "norm_projection", "residual_projection", "linear", "swiglu_block",
         "swiglu_mlp"]

SCRIPT = r"""
import json, sys
sys.path[:0] = [sys.argv[2]]
import torch
import torch.nn.functional as F
from ops import _hip
_hip.load_autograd = lambda: None
from ops import activation_execution as ae, fused_training as ft
from torch._dynamo import compiled_autograd

BF16 = torch.bfloat16

def swiglu(packed, eager=True):
    up, gate = packed.float().chunk(2, -1)
    return (F.silu(gate) * up).to(BF16)

def swiglu_backward(packed, grad, eager=True):
    up, gate = packed.float().chunk(2, -1)
    s, g = torch.sigmoid(gate), grad.float()
    return torch.cat([g * s * gate, g * up * s * (1 + gate * (1 - s))], -1).to(BF16)

def rmsnorm(x, weight, eps, eager=True):
    rstd = torch.rsqrt(x.float().square().mean(-1) + eps)
    return (x.float() * rstd[:, None] * weight).to(BF16), rstd

def rmsnorm_backward(x, weight, rstd, grad, eager=True):
    dz, r = grad.float() * weight, rstd[:, None]
    dx = dz * r - x.float() * r ** 3 * (dz * x.float()).mean(-1, keepdim=True)
    return dx.to(BF16), (grad.float() * x.float() * r).sum(0)

def mm(a, b):
    return (a.float() @ b.float()).to(BF16)

def norm_projection(x, norm_weight, weight, eps, gate_begin, gate_end):
    y, rstd = rmsnorm(x, norm_weight, eps)
    w = weight.to(BF16)
    out = mm(y, w.T)
    out[:, gate_begin:gate_end] = torch.sigmoid(out[:, gate_begin:gate_end])
    return out, rstd, y, w

def norm_projection_backward(dout, x, norm_weight, rstd, normed, w, out, gate_begin, gate_end):
    dp = dout.clone()
    s = out[:, gate_begin:gate_end]
    dp[:, gate_begin:gate_end] *= (1 - s) * s
    dx, dnorm = rmsnorm_backward(x, norm_weight, rstd, mm(dp, w))
    return dx, dnorm, mm(dp.T, normed).float()

def residual_projection(a, weight, residual):
    w = weight.to(BF16)
    return residual + mm(a, w.T), w

def linear(a, weight):
    w = weight.to(BF16)
    return mm(a, w.T), w

def linear_backward(dout, a, w):
    return mm(dout, w), mm(dout.T, a).float()

def swiglu_mlp(h, w_upgate, w_down):
    wug, wd = w_upgate.to(BF16), w_down.to(BF16)
    packed = mm(h, wug.T)
    act = swiglu(packed)
    return mm(act, wd.T), packed, act, wug, wd

def swiglu_block(h, w_upgate, w_down, residual):
    out, *rest = swiglu_mlp(h, w_upgate, w_down)
    return (residual + out, *rest)

def swiglu_block_backward(dout, h, packed, act, wug, wd):
    dpacked = swiglu_backward(packed, mm(dout, wd))
    return mm(dpacked, wug), mm(dpacked.T, h).float(), mm(dout.T, act).float()

for op, kernel in [
        (ae.bf16_swiglu, swiglu), (ae._swiglu_backward, swiglu_backward),
        (ae.bf16_rmsnorm, rmsnorm), (ae._rms_backward, rmsnorm_backward),
        (ft.fused_norm_projection, norm_projection),
        (ft.fused_norm_projection_backward, norm_projection_backward),
        (ft.fused_residual_projection, residual_projection),
        (ft.fused_residual_projection_backward, linear_backward),
        (ft.fused_linear, linear), (ft.fused_linear_backward, linear_backward),
        (ft.fused_swiglu_block, swiglu_block),
        (ft.fused_swiglu_block_backward, swiglu_block_backward),
        (ft.fused_swiglu_mlp, swiglu_mlp)]:
    op.register_kernel("cpu")(kernel)
torch.ops.load_library(sys.argv[1])

gen = torch.Generator().manual_seed(3)

def leaf(*shape, dtype=BF16):
    return torch.randn(shape, generator=gen).to(dtype).requires_grad_(True)

f32 = torch.float32
CASES = {
    "swiglu": (ae.bf16_swiglu, [leaf(6, 16)], [True]),
    "rmsnorm": (ae.bf16_rmsnorm, [leaf(6, 8), leaf(8, dtype=f32)], [1e-5, True]),
    "norm_projection": (ft.fused_norm_projection,
                        [leaf(6, 8), leaf(8, dtype=f32), leaf(24, 8, dtype=f32)], [1e-5, 8, 16]),
    "residual_projection": (ft.fused_residual_projection,
                            [leaf(6, 8), leaf(16, 8, dtype=f32), leaf(6, 16)], []),
    "linear": (ft.fused_linear, [leaf(6, 8), leaf(16, 8, dtype=f32)], []),
    "swiglu_block": (ft.fused_swiglu_block, [leaf(6, 8), leaf(32, 8, dtype=f32),
                                             leaf(8, 16, dtype=f32), leaf(6, 8)], []),
    "swiglu_mlp": (ft.fused_swiglu_mlp, [leaf(6, 8), leaf(32, 8, dtype=f32),
                                         leaf(8, 16, dtype=f32)], []),
}

def main_output(out):
    return out[0] if isinstance(out, tuple) else out

def gradients(fn, leaves, grad):
    for t in leaves:
        t.grad = None
    main_output(fn(*leaves)).backward(grad)
    return [t.grad for t in leaves]

def check(name):
    op, leaves, rest = CASES[name]
    call = lambda *args: op(*args, *rest)
    out = call(*leaves)
    node = main_output(out).grad_fn.name()
    if "GeneratedBackward" in node:
        return "the Python formula was recorded: " + node
    if name == "rmsnorm" and out[1].requires_grad:
        return "the saved statistics require a gradient"
    grad = torch.randn(main_output(out).shape, generator=gen).to(BF16)
    want = gradients(call, leaves, grad)
    if any(g is None or not g.any() for g in want):
        return "a gradient is missing"
    with compiled_autograd._enable(torch.compile(backend="aot_eager")):
        traced = gradients(call, leaves, grad)
    compiled = gradients(torch.compile(call, backend="aot_eager", fullgraph=True), leaves, grad)
    with compiled_autograd._enable(torch.compile(backend="aot_eager")):  # and both
        both = gradients(torch.compile(call, backend="aot_eager", fullgraph=True), leaves, grad)
    for label, got in (("compiled autograd", traced), ("compile", compiled), ("both", both)):
        if not all(torch.equal(a, b) for a, b in zip(want, got)):
            return label + " gives other gradients"
    return ""

for name in CASES:
    try:
        result = check(name)
    except Exception as error:
        result = type(error).__name__ + ": " + str(error)[:300]
    print(json.dumps([name, result]), flush=True)
"""


@pytest.fixture(scope="module")
def results(tmp_path_factory):
    work = tmp_path_factory.mktemp("autograd")
    source = (build_lib.CSRC / "autograd.cpp").read_text()
    assert source.count("TORCH_LIBRARY_IMPL(warpstate, AutogradCUDA") == 1
    cpu = work / "autograd_cpu.cpp"
    cpu.write_text(source.replace("TORCH_LIBRARY_IMPL(warpstate, AutogradCUDA",
                                  "TORCH_LIBRARY_IMPL(warpstate, AutogradCPU"))
    library = work / "libautograd_cpu.so"
    built = subprocess.run(build_lib.autograd_command(cpu, library), capture_output=True, text=True)
    assert built.returncode == 0, built.stderr[-2000:]
    script = work / "check.py"
    script.write_text(SCRIPT)
    run = subprocess.run([sys.executable, str(script), str(library), str(ROOT / "warpstate-ai_amd")],
                         capture_output=True, text=True, timeout=600)
    assert run.returncode == 0, run.stderr[-2000:]
    return dict(json.loads(line) for line in run.stdout.splitlines() if line.startswith("["))


@pytest.mark.parametrize("name", NAMES)
def test_backward_is_the_same_under_compiled_autograd(name, results):
    assert results[name] == ""
