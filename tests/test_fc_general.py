"""Fully connected product with a second operand of several channels on the rows kernels (csrc/fc_flex.hip): product, first derivatives
and - float32 - second ones against the oracle, at the edges of its tiles: rows around 32 and 128, contracted blocks of 16 to 80
values (in registers up to 64), columns that are no multiple of 32, one to nine channels of x2 (groups of four)."""

import copy

import pytest
import torch

from cuequivariance_amd import cue
from oracle.naive import naive_segmented_polynomial, spec_from_polynomial

pytestmark = pytest.mark.gpu
# float32: sums of up to 1 000 products of unit size, error about sqrt(1000) 2^-24 of the largest sum; bfloat16 / half: the results
# rounded once (2^-9 / 2^-12 of them), the gradients' formed factors once more
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}


def to_ir_mul(x, irreps):
    out, i = [], 0
    for mul, ir in irreps:
        out.append(x[:, i:i + mul * ir.dim].reshape(-1, mul, ir.dim).transpose(1, 2).reshape(x.shape[0], -1))
        i += mul * ir.dim
    return torch.cat(out, 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["ir_mul", "mul_ir"])
@pytest.mark.parametrize("i1,i2,io,rows", [
    ("64x0e+64x1o", "16x0e+16x1o", "64x0e+64x1o", 131),
    ("32x0e+16x1o", "4x0e+3x1o", "48x0e+32x1o", 33),
    ("32x0e+32x1o", "9x0e+5x1o", "16x0e+64x1o+16x1e", 1),
    ("48x0e+16x1o+32x2e", "2x0e+1x1o+5x2e", "32x0e+16x1o+48x2e", 70),
    ("80x0e+32x1o", "9x0e+2x1o", "16x0e+80x1o+16x1e", 29),
])
def test_product_and_derivatives(device, dtype, layout, i1, i2, io, rows):
    from cuequivariance_amd import cuet

    i1, i2, io = cue.Irreps("O3", i1), cue.Irreps("O3", i2), cue.Irreps("O3", io)
    m = copy.deepcopy(cuet.FullyConnectedTensorProduct(i1, i2, io, layout=getattr(cue, layout), internal_weights=False))
    g = torch.Generator().manual_seed(rows)
    r = lambda *shape: torch.randn(*shape, dtype=torch.float64, generator=g).to(dtype).double()
    args = [r(1, m.weight_numel), r(rows, i1.dim), r(rows, i2.dim)]
    cot, second = r(rows, io.dim), [r(*t.shape) for t in args]
    into = (lambda t, irreps: to_ir_mul(t, irreps)) if layout == "mul_ir" else (lambda t, irreps: t)
    spec = spec_from_polynomial(m.f._polynomial_orig)

    def derivatives(f, args, cot, second):
        args, cot = [t.clone().requires_grad_(True) for t in args], cot.clone().requires_grad_(True)
        out = f(*args)
        assert out is not None
        plain = torch.autograd.grad(out, args, cot, retain_graph=True)
        first = torch.autograd.grad(out, args, cot, create_graph=True)
        return [out, *plain, *torch.autograd.grad(first, [*args, cot], second)]

    want = derivatives(lambda w, a, b: naive_segmented_polynomial(spec, [w, a, b])[0], [args[0], into(args[1], i1), into(args[2], i2)], into(cot, io),
                       [second[0], into(second[1], i1), into(second[2], i2)])
    to = lambda t: t.to(dtype).to(device)
    assert m.general(to(args[0]), to(args[1]), to(args[2])) is not None  # (these kernels, not the stage in memory)
    got = derivatives(lambda w, a, b: m(a, b, w), [to(t) for t in args], to(cot), [to(t) for t in second])
    for k, (a, b, irreps) in enumerate(zip(got, want, [io, None, i1, i2, None, i1, i2, io])):
        a = a.detach().cpu().double()
        a = a if irreps is None else into(a, irreps)
        assert (a - b.detach()).abs().max().item() <= TOL[dtype] * b.abs().max().item(), k


def test_calls_it_leaves_to_the_other_ways(device):
    """64-bit rows, one row against many and other types of weights keep the stage that forms the products in memory."""
    from cuequivariance_amd import cuet

    i1, i2 = cue.Irreps("O3", "32x0e+32x1o"), cue.Irreps("O3", "4x0e+4x1o")
    m = cuet.FullyConnectedTensorProduct(i1, i2, i1, layout=cue.ir_mul, internal_weights=False)
    r = lambda *shape: torch.randn(*shape, dtype=torch.float64, device=device)
    w, a, b = r(1, m.weight_numel), r(7, i1.dim), r(7, i2.dim)
    assert m.general(w, a, b) is None and m.general(w.float(), a.float(), b[:1].float()) is None and m.general(w.float(), a.bfloat16(), b.bfloat16()) is None
    want = m(a, b, w)
    torch.testing.assert_close(m(a.float(), b.float(), w.float()).double(), want, rtol=1e-5, atol=1e-5 * want.abs().max().item())
    torch.testing.assert_close(m(a.float(), b[:1].float(), w.float()).double(), m(a, b[:1].expand(7, -1), w), rtol=1e-5, atol=1e-5 * want.abs().max().item())


def test_long_blocks_go_by_rows_and_channels(device):
    """Blocks of more than 64 values: 2-byte rows up to 4 000, at most 16 values of the second operand."""
    from cuequivariance_amd import cuet

    for second, rows, dtype, taken in (("10x0e", 4000, torch.bfloat16, True), ("10x0e", 4001, torch.bfloat16, False), ("10x0e", 4001, torch.float32, True),
                                       ("17x0e", 5, torch.float32, False)):
        i1, i2 = cue.Irreps("O3", "96x0e"), cue.Irreps("O3", second)
        m = cuet.FullyConnectedTensorProduct(i1, i2, i1, layout=cue.ir_mul, internal_weights=False)
        w, a, b = (torch.randn(*s, device=device, dtype=dtype) for s in ((1, m.weight_numel), (rows, i1.dim), (rows, i2.dim)))
        assert (m.general(w, a, b) is not None) == taken
        want = torch.einsum("zu,zv,uvw->zw", a[-4:].double(), b[-4:].double(), w.double().reshape(96, i2.dim, 96)) / (96 * i2.dim) ** 0.5
        torch.testing.assert_close(m(a, b, w)[-4:].double(), want, rtol=0, atol=(1e-5 if dtype == torch.float32 else 1e-2) * want.abs().max().item())
