"""The native autograd kernels of the row and fused training operators record what their
Python formulas record: gradients, auxiliary outputs, create_graph and saved-tensor hooks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(name):
    from ops import activation_execution as ae, fused_training as ft

    gen = torch.Generator("cuda").manual_seed(5)

    def leaf(*shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=gen, device="cuda").to(dtype).requires_grad_(True)

    f32 = torch.float32
    x, w = leaf(72, 64), leaf(64, dtype=f32)
    if name == "swiglu":
        return ae.bf16_swiglu, [leaf(72, 128)], [True]
    if name == "rmsnorm":
        return ae.bf16_rmsnorm, [x, w], [1e-5, False]
    if name == "norm_projection":
        return ft.fused_norm_projection, [x, w, leaf(320, 64, dtype=f32)], [1e-5, 192, 256]
    if name == "residual_projection":
        return ft.fused_residual_projection, [x, leaf(96, 64, dtype=f32), leaf(72, 96)], []
    if name == "linear":
        return ft.fused_linear, [x, leaf(96, 64, dtype=f32)], []
    if name == "swiglu_block":
        return ft.fused_swiglu_block, [x, leaf(256, 64, dtype=f32), leaf(64, 128, dtype=f32),
                                       leaf(72, 64)], []
    return ft.fused_swiglu_mlp, [x, leaf(256, 64, dtype=f32), leaf(64, 128, dtype=f32)], []


NAMES = ["swiglu", "rmsnorm", "norm_projection", "residual_projection", "linear", "swiglu_block",
         "swiglu_mlp"]


@pytest.mark.parametrize("name", NAMES)
def test_native_kernels_match_the_python_formulas(name):
    op, leaves, rest = _case(name)
    out = op(*leaves, *rest)
    outs = out if isinstance(out, tuple) else (out,)
    grad = torch.randn_like(outs[0])
    got = torch.autograd.grad(outs[0], leaves, grad, retain_graph=True)
    # The Python formula, through the operator's registered backward.
    ctx = type("Ctx", (), {})()
    ctx.save_for_backward = lambda *t: setattr(ctx, "saved_tensors", t)
    ctx.mark_non_differentiable = lambda *t: None
    op._setup_context_fn(ctx, (*leaves, *rest), out)
    with torch.no_grad():
        want = op._backward_fn(ctx, grad, *[None] * (len(outs) - 1))
    for g, e in zip(got, want):
        assert torch.equal(g, e), name
    # Only auxiliary outputs differentiated: the main output's gradient is zero.
    if len(outs) > 2:
        zero = torch.autograd.grad(outs[-1].float().sum(), leaves, retain_graph=True,
                                   allow_unused=True)
        assert all(g is None or not g.any() for g in zero), name
    # create_graph works; the gradient itself cannot be differentiated.
    again = torch.autograd.grad(outs[0], leaves, grad, create_graph=True)
    assert torch.equal(again[0], got[0])
    with pytest.raises(RuntimeError, match="no autograd formula"):
        torch.autograd.grad(again[0].float().sum(), leaves)


@pytest.mark.parametrize("name", NAMES)
def test_saved_tensor_hooks_see_every_saved_tensor(name):
    op, leaves, rest = _case(name)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        out = op(*leaves, *rest)
    first = out[0] if isinstance(out, tuple) else out
    grad = torch.randn_like(first)
    plain = op(*leaves, *rest)
    plain = plain[0] if isinstance(plain, tuple) else plain
    for g, e in zip(torch.autograd.grad(first, leaves, grad),
                    torch.autograd.grad(plain, leaves, grad)):
        assert torch.equal(g, e), name
    assert packed


@pytest.mark.parametrize("name", NAMES)
def test_calls_that_record_nothing_take_forward_mode_tensors(name):
    import torch.autograd.forward_ad as fwad

    op, leaves, rest = _case(name)
    want = op(*leaves, *rest)
    want = want[0] if isinstance(want, tuple) else want
    plain = [t.detach() for t in leaves]
    with fwad.dual_level():
        got = op(fwad.make_dual(plain[0], torch.ones_like(plain[0])), *plain[1:], *rest)
        got = got[0] if isinstance(got, tuple) else got
        primal, tangent = fwad.unpack_dual(got)
        assert tangent is None and not primal.requires_grad
        assert torch.equal(primal, want.detach())


@pytest.mark.parametrize("name", NAMES)
def test_compiled_autograd_traces_the_native_nodes(name):
    """A backward under compiled autograd, of an eager and of a compiled call, gives the
    eager gradients."""
    from torch._dynamo import compiled_autograd

    op, leaves, rest = _case(name)

    def call(*inputs):
        out = op(*inputs, *rest)
        return out[0] if isinstance(out, tuple) else out

    def gradients(fn, grad):
        for t in leaves:
            t.grad = None
        fn(*leaves).backward(grad)
        return [t.grad for t in leaves]

    torch._dynamo.reset()
    try:
        out = call(*leaves)
        assert "Generated" not in out.grad_fn.name()  # the C++ node, not the Python formula's
        grad = torch.randn_like(out)
        want = gradients(call, grad)
        for fn in (call, torch.compile(call, backend="aot_eager", fullgraph=True)):
            with compiled_autograd._enable(torch.compile(backend="aot_eager")):
                got = gradients(fn, grad)
            assert all(torch.equal(a, b) for a, b in zip(want, got)), name
    finally:
        torch._dynamo.reset()
