"""The fully connected product on its table-driven kernels (few rows, extents the generated kernels do not take) and with the weight
gradient's factors through memory (many rows): product, first derivatives and - float32 - second ones against the oracle."""

import pytest
import torch

from cuequivariance_amd import cue
from oracle.naive import naive_segmented_polynomial, spec_from_polynomial

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}


def to_ir_mul(x, irreps):
    out, i = [], 0
    for mul, ir in irreps:
        out.append(x[:, i:i + mul * ir.dim].reshape(-1, mul, ir.dim).transpose(1, 2).reshape(x.shape[0], -1))
        i += mul * ir.dim
    return torch.cat(out, 1)


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["ir_mul", "mul_ir"])
@pytest.mark.parametrize("i1,i2,io,rows", [
    ("128x0e+128x1o", "0e+1o", "128x0e+128x1o", 33),
    ("16x0e+48x1o+32x2e", "0e+1o+2e", "32x0e+16x1o+48x2e", 70),
    ("32x1o", "1o", "64x0e", 1),
])
def test_product_and_derivatives(device, dtype, layout, i1, i2, io, rows, tiled):
    from cuequivariance_amd import cuet

    i1, i2, io = cue.Irreps("O3", i1), cue.Irreps("O3", i2), cue.Irreps("O3", io)
    m = cuet.FullyConnectedTensorProduct(i1, i2, io, layout=getattr(cue, layout), internal_weights=False)
    dense = (m.f_rows if m.f_rows is not None else m.f).m.dense
    op = dense.fully_connected
    assert op is not None and dense.fc_takes(torch.empty(0, dtype=dtype), ())
    if tiled:
        from cuequivariance_amd.cuet.dense import _fc_tables

        fresh = _fc_tables(dense)
        op = type(op)(dense.input_sizes[1], dense.input_sizes[2], dense.out_size, dense.input_sizes[0], dense.rows_mul_ir, dense.dx1_covers_input,
                      dense.fwd_covers_output, fresh[2], fresh[3], fresh[0], fresh[1])
        op.add_tiled_dw(fresh[4], 0, 0)
        dense._fc = {on: op for on in (True, False)}
    g = torch.Generator().manual_seed(rows)
    r = lambda *shape: torch.randn(*shape, dtype=torch.float64, generator=g).to(dtype).double()
    args = [r(1, m.weight_numel), r(rows, i1.dim), r(rows, i2.dim)]
    cot, second = r(rows, io.dim), [r(*t.shape) for t in args]
    into = (lambda t, irreps: to_ir_mul(t, irreps)) if layout == "mul_ir" else (lambda t, irreps: t)
    spec = spec_from_polynomial(m.f._polynomial_orig if m.f is not None else m.f_per_sample._polynomial)

    def derivatives(f, args, cot, second):
        args, cot = [t.clone().requires_grad_(True) for t in args], cot.clone().requires_grad_(True)
        out = f(*args)
        plain = torch.autograd.grad(out, args, cot, retain_graph=True)
        first = torch.autograd.grad(out, args, cot, create_graph=True)
        return [out, *plain, *torch.autograd.grad(first, [*args, cot], second)]

    want = derivatives(lambda w, a, b: naive_segmented_polynomial(spec, [w, a, b])[0], [args[0], into(args[1], i1), args[2]], into(cot, io),
                       [second[0], into(second[1], i1), second[2]])
    to = lambda t: t.to(dtype).to(device)
    got = derivatives(lambda w, a, b: m(a, b, w), [to(t) for t in args], to(cot), [to(t) for t in second])
    for k, (a, b, irreps) in enumerate(zip(got, want, [io, None, i1, None, None, i1, None, io])):
        a = a.detach().cpu().double()
        a = a if irreps is None else into(a, irreps)
        assert (a - b.detach()).abs().max().item() <= TOL[dtype] * b.abs().max().item(), k
