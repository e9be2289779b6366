"""Capture of kernels that have not run before: the macro-tile, and with it the kernel, follows
the sizes, so a graph of other sizes than the warm-up's may hold a kernel's first launch. In a
process of its own, where nothing has run."""
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu
PACKAGE = Path(__file__).resolve().parents[1] / "warpstate-ai_amd"
SCRIPT = """
import sys
sys.path.insert(0, sys.argv[1])
import torch
from ops import fused_execution as fx
from ops.matmul_epilogue import launch_swiglu_mm

def ints(*shape):
    return torch.randint(-2, 3, shape, device="cuda").bfloat16()

def make_step(m, n, k):
    a, w, r, dy = ints(m, k), ints(n, k), ints(m, n), ints(m, n)
    norm = torch.ones(k, device="cuda")
    def step():
        gate, _ = fx.rmsnorm_gate_mm(a, norm, 1e-5, w, (0, 16))
        packed, act = launch_swiglu_mm(a, w.T, "persistent", (128, 128, 32, 8, 3), True)
        return (fx.mm(a, w.T), fx.residual_mm(a, w, r), fx.dgrad_mm(dy, w), fx.mm_f32(dy.T, a),
                packed, act, gate)
    return step

make_step(16384, 2048, 2048)()
torch.cuda.synchronize()
for shape in ((512, 1280, 1280), (1992, 1280, 4480), (1024, 4096, 256)):
    step = make_step(*shape)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    want = step()
    for _ in range(2):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(out, want)), shape
    print(shape, "ok", flush=True)
"""


def test_capture_at_sizes_that_have_not_run():
    run = subprocess.run([sys.executable, "-c", SCRIPT, str(PACKAGE)], capture_output=True,
                         text=True, timeout=100)
    assert run.returncode == 0, run.stdout + run.stderr[-2000:]
    assert run.stdout.count("ok") == 3
