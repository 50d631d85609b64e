"""Long runs whose length is no multiple of a 16-byte vector: whole vectors between the boundaries
inside a chunk, single elements around them.  The same tensors one element off alignment go element
by element, so outputs and input gradients are equal bit for bit, and the encoding gradients (fp64
sums in another order, rounded to fp32 once) within one unit in the last place."""
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


def _off(t):
    """The same values, starting one element past an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.flatten()
    return buf[1:].view(t.shape)


# runs below one vector, at a chunk's edge (4096 fp32, 8192 16-bit, 2048 fp64 elements) and across
# several, every misalignment of a row's start, and two chunks per workgroup (over 2048 chunks)
@pytest.mark.parametrize("shape,enc", [
    ((1,), ()), ((7,), ()), ((9,), ()), ((4095,), ()), ((4097,), ()), ((8191,), ()), ((8193,), ()),
    ((9, 1025), (9, 1)), ((17, 4099), (17, 1)), ((9, 8185), (9, 1)), ((1030, 8197), (1030, 1)),
    ((4099, 4101), ())])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_vectors_and_edges_equal_single_elements(cuda, shape, enc, dtype):
    gen = torch.Generator(device=cuda).manual_seed(len(shape) * 7919 + shape[-1])
    x = torch.randn(shape, generator=gen, device=cuda).to(dtype)
    g = torch.randn(shape, generator=gen, device=cuda).to(dtype)
    res = []
    for form in (lambda t: t, _off):
        xf = form(x.detach()).requires_grad_()
        s = torch.full(enc, 0.013, device=cuda).requires_grad_()
        o = torch.full(enc, 3.0, device=cuda).requires_grad_()
        y = Q.quantize_dequantize(xf, s, o, -128, 127)
        y.backward(form(g))
        lo, hi = Q.minmax(xf.detach(), enc)
        res.append((y.detach(), xf.grad, s.grad, o.grad, lo, hi))
    a, b = res
    for k in (0, 1, 4, 5):
        assert torch.equal(a[k], b[k]), k
    for k in (2, 3):
        # one unit where the value stands, and the sums' own error (2^-52 of the terms' magnitudes)
        terms = (g.double().abs() * 128).sum() * 2.0 ** -40
        assert bool(((a[k] - b[k]).abs().double() <= a[k].abs().double() * 2.0 ** -23 + terms).all())


# One check for the quotients of a vector: zeros of either sign, values outside the range of the
# residual steps, infinities and NaN, one in a vector or all of it, and scales outside theirs.
SCALES = [0.013, 2.0 ** -61, 2.0 ** 61, 2.0 ** -60, 2.0 ** 60, 1e-39, 0.0]


def _special_vectors(cuda, dtype):
    gen = torch.Generator(device=cuda).manual_seed(11)
    special = torch.tensor([0.0, -0.0, 2.0 ** -40, -2.0 ** -41, 2.0 ** 40, -2.0 ** 41, 1e-45, 3e38,
                            float("inf"), -float("inf"), float("nan"), 6.5e4], device=cuda)
    x = torch.randn(64, 8, 8, generator=gen, device=cuda)
    x[1:49, :, 3] = special.repeat_interleave(4)[:, None]       # one of a vector
    x[49:61] = special[:, None, None]                           # all of it
    x = x.flatten().to(dtype)
    return x, torch.randn(x.shape, generator=gen, device=cuda).to(dtype)


def _bits(t):
    return t.detach().view(torch.int32 if t.dtype == torch.float32 else torch.int16)


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_quotients_of_a_vector_equal_single_ones(cuda, scale, dtype):
    x, g = _special_vectors(cuda, dtype)
    res = []
    for form in (lambda t: t, _off):
        xf = form(x.detach()).requires_grad_()
        s = torch.tensor(scale, device=cuda).requires_grad_()
        o = torch.tensor(0.0, device=cuda).requires_grad_()
        y = Q.quantize_dequantize(xf, s, o, -128, 127)
        y.backward(form(g))
        res.append([_bits(t) for t in (y, xf.grad)])
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_codes_of_a_vector_equal_single_ones(cuda, scale, dtype):
    """Quantization, whose quotients of a 16-bit vector share the check too, and its backward."""
    x, g = _special_vectors(cuda, dtype)
    res = []
    for form in (lambda t: t, _off):
        xf = form(x.detach()).requires_grad_()
        s = torch.tensor(scale, device=cuda).requires_grad_()
        q = Q.quantize(xf, s, torch.tensor(0.0, device=cuda), -128, 127)
        q.backward(form(g.to(q.dtype)))
        res.append([_bits(t) for t in (q, xf.grad)])
    for a, b in zip(*res):
        assert torch.equal(a, b)
