"""Fully connected products on either side of the row counts up to which the wavefronts of a workgroup share a tile
(``cueq_fc_flex``): the last rows of the shared and of the unshared kernels against 64 bits, with finite operands and with an
infinite component (which the shared tile hands to the loop over coupled components as a whole)."""

import pytest
import torch

from cuequivariance_amd import cue
from tests.test_fc_infinities import reference

pytestmark = pytest.mark.gpu


# two column tiles a row tile: 3 x 256 tiles of float, 2 x 256 of packed 2-byte weights; fewer parts than wavefronts in the first
@pytest.mark.parametrize("infinite", [False, True])
@pytest.mark.parametrize("i1,i2,rows,dtype", [
    ("32x0e+32x1o", "0e+1o", 45, torch.float32), ("32x0e+32x1o", "3x0e+3x1o", 12_288, torch.float32), ("32x0e+32x1o", "3x0e+3x1o", 12_289, torch.float32),
    ("32x0e+32x1o", "5x0e+5x1o", 8_192, torch.bfloat16), ("32x0e+32x1o", "5x0e+5x1o", 8_193, torch.bfloat16),
    ("64x0e+64x1o", "3x0e+3x1o", 31, torch.float16), ("48x0e+48x1o+16x2e", "3x0e+2x2e", 65, torch.float32), ("48x0e+48x1o+16x2e", "3x0e+2x2e", 65, torch.bfloat16)])
@pytest.mark.parametrize("layout", [cue.ir_mul, cue.mul_ir])
def test_values_and_gradients(device, layout, i1, i2, rows, dtype, infinite):
    from cuequivariance_amd import cuet

    i1, i2 = cue.Irreps("O3", i1), cue.Irreps("O3", i2)
    m = cuet.FullyConnectedTensorProduct(i1, i2, i1, layout=layout, internal_weights=False)
    e = cue.descriptors.fully_connected_tensor_product(i1, i2, i1)
    g = torch.Generator(device=device).manual_seed(rows)
    r = lambda *shape: torch.randn(*shape, generator=g, device=device).to(dtype)
    w, x1, x2, cot = r(1, m.weight_numel), r(rows, i1.dim), r(rows, i2.dim), r(rows, i1.dim)
    if infinite:
        x1[rows - 1, i1[0].mul + 1] = float("inf")  # (ir_mul: component 0, mul_ir: component 1 of the vectors)

    def rows_of(t, irreps, back=False):  # rows of the layout <-> ir_mul
        out, at = [], 0
        for mul, ir in irreps if layout == cue.mul_ir else ():
            b = t[:, at: at + mul * ir.dim]
            out.append((b.reshape(-1, ir.dim, mul) if back else b.reshape(-1, mul, ir.dim)).transpose(1, 2).reshape(t.shape[0], -1))
            at += mul * ir.dim
        return torch.cat(out, 1) if out else t

    ref = [t.double().requires_grad_() for t in (w, rows_of(x1, i1), rows_of(x2, i2))]
    want = reference(e, *ref)
    dw, d1, d2 = torch.autograd.grad(want, ref, rows_of(cot, i1).double())
    got_in = [t.requires_grad_() for t in (x1, x2, w)]
    out = m(*got_in)
    g1, g2, gw = torch.autograd.grad(out, got_in, cot)
    for name, a, b in (("out", rows_of(out.detach(), i1), want), ("dx1", rows_of(g1, i1), d1), ("dx2", rows_of(g2, i2), d2), ("dw", gw, dw)):
        a, b = a.double(), b.detach()
        keep = torch.isfinite(b)
        assert keep.any() or name == "dw"
        assert torch.isfinite(a[keep]).all(), name
        # (float32 sums of up to some 20 000 products; 2-byte results rounded once, formed factors once more)
        tol = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}[dtype]
        if keep.any():
            assert (a[keep] - b[keep]).abs().max().item() <= tol * b[keep].abs().max().item(), name


# as many tiles as are shared, and one row more: no sharing of single parts, otherwise 1, 2 and 6 tiles a CU by 2, 6 and 32 parts of a block;
# with blocks of five components 2 and 12 by 3 and 7 (256 CUs; two or three column tiles a row tile)
@pytest.mark.parametrize("i1,i2,rows,most", [
    ("32x0e+32x1o", "0e", 31, 0), ("32x0e+32x1o", "0e+1o", 4_097, 4_096), ("32x0e+32x1o", "3x0e+3x1o", 8_193, 8_192),
    ("32x0e+32x1o", "16x0e+16x1o", 24_577, 24_576), ("32x0e+32x1o+32x2e", "0e+1o+2e", 5_441, 5_440), ("32x0e+32x1o+32x2e", "2x0e+2x1o+2x2e", 32_769, 32_768)])
def test_which_tiles_are_shared(device, i1, i2, rows, most):
    from cuequivariance_amd import _lib

    for n in (rows, most) if most else (rows,):
        _lib.timing_begin()
        try:
            test_values_and_gradients(device, cue.ir_mul, i1, i2, n, torch.float32, False)
        finally:
            labels = {k for k in _lib.timing_end() if k.startswith(("fc_flex_fwd", "fc_flex_dx"))}
        assert labels == ({"fc_flex_fwd_shared", "fc_flex_dx_shared"} if n <= most else {"fc_flex_fwd", "fc_flex_dx"}), (n, labels)
