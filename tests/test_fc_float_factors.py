"""Fully connected products of 2-byte rows whose other form is float32 throughout (half; bfloat16 with few scalar paths): the weight
gradient's factors ``sum_jk C x2 g`` must not be rounded to the rows' type, nor leave its range, and half operands are exact."""

import pytest
import torch

from cuequivariance_amd import cue
from oracle.naive import naive_segmented_polynomial, spec_from_polynomial

pytestmark = pytest.mark.gpu
SMALL, LARGE = ("32x0e+32x1o", "4x0e+4x1o", "32x0e+32x1o"), ("64x0e+64x1o", "16x0e+16x1o", "64x0e+64x1o")
TINY, ONE = ("16x0e+16x1o", "2x0e+2x1o", "16x0e+16x1o"), ("96x0e+96x1o", "0e+1o", "96x0e+96x1o")


def setup(irreps, rows, dtype, layout, scales):
    from cuequivariance_amd import cuet

    irreps = [cue.Irreps("O3", i) for i in irreps]
    m = cuet.FullyConnectedTensorProduct(*irreps, layout=getattr(cue, layout), internal_weights=False)
    g = torch.Generator().manual_seed(rows)
    shapes = (1, m.weight_numel), (rows, irreps[0].dim), (rows, irreps[1].dim), (rows, irreps[2].dim)
    return m, irreps, [(torch.randn(*s, dtype=torch.float64, generator=g) * f).to(dtype) for s, f in zip(shapes, scales)]


def exact(m, irreps, tensors, layout):
    """(out, dw) in float64."""
    w, x1, x2, g = (t.double() for t in tensors)
    if layout == "mul_ir":
        def lie(x, irreps, back=False):
            out, i = [], 0
            for mul, ir in irreps:
                b = x[:, i:i + mul * ir.dim]
                out.append((b.reshape(-1, ir.dim, mul) if back else b.reshape(-1, mul, ir.dim)).transpose(1, 2).reshape(x.shape[0], -1))
                i += mul * ir.dim
            return torch.cat(out, 1)
        x1, x2, g = lie(x1, irreps[0]), lie(x2, irreps[1]), lie(g, irreps[2])
    w.requires_grad_(True)
    out = naive_segmented_polynomial(spec_from_polynomial(m.f._polynomial_orig), [w, x1, x2])[0]
    dw, = torch.autograd.grad(out, w, g)
    return (lie(out.detach(), irreps[2], True) if layout == "mul_ir" else out.detach()), dw


def rounded_once(got, want, dtype):
    """The error is that of one rounding to the type (float32 sums of a few thousand products add about 1e-6)."""
    error = lambda t: ((t.double() - want).norm() / want.norm()).item()
    assert torch.isfinite(got).all()
    assert error(got.cpu()) <= 1.1 * error(want.to(dtype)) + 1e-6, (error(got.cpu()), error(want.to(dtype)))


@pytest.mark.parametrize("layout", ["ir_mul", "mul_ir"])
@pytest.mark.parametrize("irreps,rows,dtype", [
    (SMALL, 300, torch.bfloat16), (TINY, 300, torch.bfloat16), (SMALL, 300, torch.float16), (LARGE, 130, torch.float16), (ONE, 300, torch.float16),
    (ONE, 14_000, torch.float16),  # (factors through memory)
])
def test_weight_gradient_is_rounded_once(device, irreps, rows, dtype, layout):
    m, irreps, t = setup(irreps, rows, dtype, layout, (1, 1, 1, 1))
    out, dw = exact(m, irreps, t, layout)
    w, x1, x2, g = (v.to(device) for v in t)
    w.requires_grad_(True)
    got = m(x1, x2, w)
    rounded_once(got.detach(), out, dtype)
    rounded_once(torch.autograd.grad(got, w, g)[0], dw, dtype)


@pytest.mark.parametrize("irreps", [ONE, LARGE])
def test_factors_beyond_the_range_of_half(device, irreps):
    m, irreps, t = setup(irreps, 40, torch.float16, "ir_mul", (1e-3, 2e-4, 100, 1e4))  # factors of some 2e5, gradients of some 1e3
    dw = exact(m, irreps, t, "ir_mul")[1]
    w, x1, x2, g = (v.to(device) for v in t)
    w.requires_grad_(True)
    rounded_once(torch.autograd.grad(m(x1, x2, w), w, g)[0], dw, torch.float16)


@pytest.mark.parametrize("irreps", [ONE, LARGE])
def test_operands_below_the_normal_range_of_half(device, irreps):
    m, irreps, t = setup(irreps, 40, torch.float16, "ir_mul", (2.0 ** 8, 2.0 ** -17, 1, 2.0 ** 8))
    out, dw = exact(m, irreps, t, "ir_mul")
    w, x1, x2, g = (v.to(device) for v in t)
    w.requires_grad_(True)
    got = m(x1, x2, w)
    rounded_once(got.detach(), out, torch.float16)
    rounded_once(torch.autograd.grad(got, w, g)[0], dw, torch.float16)
