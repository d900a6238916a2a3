"""Linear on the launches for few rows and for shapes the row-streaming launches do not take: several input blocks per output
block, extents beyond 128 and between the tile sizes, ragged rows, both row orders, all first derivatives and, in float32, the
second ones against the oracle."""

import pytest
import torch

from cuequivariance_amd import cue
from oracle.naive import naive_segmented_polynomial, spec_from_polynomial

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}


def to_ir_mul(x, irreps):
    out, i = [], 0
    for mul, ir in irreps:
        b = x[:, i:i + mul * ir.dim].reshape(-1, mul, ir.dim)
        out.append(b.transpose(1, 2).reshape(x.shape[0], -1))
        i += mul * ir.dim
    return torch.cat(out, 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["ir_mul", "mul_ir"])
@pytest.mark.parametrize("irreps_in,irreps_out,rows", [
    ("32x0e+32x0e+32x1o+32x1o+64x1o", "64x0e+32x1o", 1),          # sums over input blocks, one row
    ("128x0e+192x1o+192x2e", "64x0e+64x1o+64x2e", 33),            # contraction beyond 128
    ("48x0e+16x1o+80x2e+16x3o", "16x0e+48x1o+16x2e+16x3o", 70),   # column tiles partly filled, 7 components
    ("64x0e+64x1o", "64x0e+64x0e+64x1o", 257),                    # two output blocks from one input block
])
def test_linear_against_the_oracle(device, dtype, layout, irreps_in, irreps_out, rows):
    from cuequivariance_amd import cuet

    irreps_in, irreps_out = cue.Irreps("O3", irreps_in), cue.Irreps("O3", irreps_out)
    m = cuet.Linear(irreps_in, irreps_out, layout=getattr(cue, layout), internal_weights=False, method="fused_tp")
    op = m._linear_op()
    assert op is not None and op.takes(torch.empty(0, dtype=dtype))
    g = torch.Generator().manual_seed(rows)
    r = lambda *shape: torch.randn(*shape, dtype=torch.float64, generator=g).to(dtype).double()
    w, x, cot, dw, dx = r(1, m.weight_numel), r(rows, irreps_in.dim), r(rows, irreps_out.dim), r(1, m.weight_numel), r(rows, irreps_in.dim)
    into = (lambda t, irreps: to_ir_mul(t, irreps)) if layout == "mul_ir" else (lambda t, irreps: t)
    spec = spec_from_polynomial(m.f._polynomial_orig)

    def derivatives(f, w, x, cot, dw, dx):
        w, x, cot = w.clone().requires_grad_(True), x.clone().requires_grad_(True), cot.clone().requires_grad_(True)
        out = f(w, x)
        first = torch.autograd.grad(out, [w, x], cot, create_graph=True)
        second = torch.autograd.grad(first, [w, x, cot], [dw, dx])
        return [out, *first, *second]

    want = derivatives(lambda a, b: naive_segmented_polynomial(spec, [a, b])[0], w, into(x, irreps_in), into(cot, irreps_out), dw, into(dx, irreps_in))
    got = derivatives(lambda a, b: m(b, a), *[t.to(dtype).to(device) for t in (w, x, cot, dw, dx)])
    rows_of = [irreps_out, None, irreps_in, None, irreps_in, irreps_out]
    for k, (a, b, irreps) in enumerate(zip(got, want, rows_of)):
        a = a.detach().cpu().double()
        a = a if irreps is None else into(a, irreps)
        assert a.shape == b.shape
        assert (a - b.detach()).abs().max().item() <= TOL[dtype] * b.abs().max().item(), k
