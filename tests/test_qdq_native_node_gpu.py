"""The C++ autograd node of the learnable min / max path against the Python Function it stands in
for: the same kernels on the same operands, so outputs and gradients are equal bit for bit."""
import sys
from pathlib import Path

import pytest
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "rx-met_amd"))
import mi355x_qdq as Q  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cuda():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda:0")


# (shape, encoding shape, block, form of the input, form of the gradient)
CASES = [
    ((64, 576), (64, 1), None, "plain", "plain"),
    ((3, 5, 7), (), None, "plain", "expanded"),
    ((33, 65), (65,), None, "transposed", "transposed"),
    ((12, 48), (12, 3), (1, 16), "plain", "transposed"),
    ((2, 3, 4, 5), (2, 1, 4, 1), None, "channels_last", "plain"),
    ((2, 3, 4, 5, 2), (2, 1, 4, 1, 2), None, "plain", "plain"),  # permuted layout
    ((1, 1), (1, 1), None, "plain", "plain"),
    ((40, 30), (40, 1), None, "offset", "offset"),  # misaligned start
]


def _form(t, form):
    if form == "transposed":
        return t.transpose(-1, -2).contiguous().transpose(-1, -2)
    if form == "channels_last":
        return t.contiguous(memory_format=torch.channels_last)
    if form == "offset":
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    if form == "expanded":
        return t.flatten()[:1].expand(t.numel()).view(t.shape) if t.numel() == 1 else \
            t.flatten()[0].expand(t.shape)
    return t


@pytest.mark.parametrize("need", ["all", "no_x", "min_only"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-{c[1]}-{c[3]}-{c[4]}" for c in CASES])
def test_native_node_equals_python_function(cuda, monkeypatch, case, dtype, need):
    shape, enc, block, xform, gform = case
    gen = torch.Generator().manual_seed(len(shape))
    x0 = _form(torch.randn(shape, generator=gen).to(dtype).to(cuda), xform)
    g0 = _form(torch.randn(shape, generator=gen).to(dtype).to(cuda), gform)
    mn0 = -torch.rand(enc, generator=gen).to(cuda) - 0.2
    mx0 = torch.rand(enc, generator=gen).to(cuda) + 0.2

    def run():
        x = x0.detach().clone(memory_format=torch.preserve_format)
        x = _form(x, xform).requires_grad_(need != "no_x")
        mn = mn0.clone().requires_grad_(True)
        mx = mx0.clone().requires_grad_(need != "min_only")
        y = Q.quantize_dequantize_minmax(x, mn, mx, -8, 7, False, 1e-8, 0.0, block, 0.0)
        name = type(y.grad_fn).__name__
        y.backward(g0)
        return name, [y.detach(), x.grad, mn.grad, mx.grad]

    name, got = run()
    monkeypatch.setattr(Q, "_native_node", lambda *t: False)
    ref_name, exp = run()
    assert (name != ref_name) == (xform in ("plain", "offset") and len(shape) != 5)
    for a, e in zip(got, exp):
        assert (a is None) == (e is None)
        if a is not None:
            assert a.shape == e.shape and a.dtype == e.dtype and a.stride() == e.stride()
            assert torch.equal(a, e)


def test_native_node_keeps_autograd_rules(cuda):
    """Saved-tensor hooks see the saved tensors, a changed operand is refused in the backward, a
    second backward and forward mode are refused, another stream gives the same gradients."""
    x = torch.randn(64, 96, device=cuda, requires_grad=True)
    mn = torch.full((64, 1), -1.0, device=cuda, requires_grad=True)
    mx = torch.full((64, 1), 1.5, device=cuda, requires_grad=True)

    def f(x):
        return Q.quantize_dequantize_minmax(x, mn, mx, -8, 7, False, 1e-8, 0.0, None, 0.0)

    def grads(y):
        return torch.autograd.grad(y, (x, mn, mx), torch.ones_like(y) * 0.5)

    ref = grads(f(x))
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(
            lambda t: (seen.append(tuple(t.shape)), t.cpu())[1], lambda t: t.to(cuda)):
        y = f(x)
    assert seen == [(64, 96), (64, 1), (64, 1)]
    assert all(torch.equal(a, b) for a, b in zip(grads(y), ref))
    with pytest.raises(RuntimeError, match="second time"):
        grads(y)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = grads(f(x))
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(other, ref))
    y = f(x)
    with torch.no_grad():
        mn.mul_(1.0)
    with pytest.raises(RuntimeError, match="inplace"):
        grads(y)
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        f(fwAD.make_dual(x.detach().requires_grad_(), torch.ones_like(x)))
    with pytest.raises(RuntimeError):
        torch.func.vmap(f)(x[None])
