"""Fully connected products with one infinite component: only what the Clebsch-Gordan coefficients couple to it may be infinite or NaN -
a structural zero of the coefficients is no factor of 0 (``0 * inf``)."""

import pytest
import torch

from cuequivariance_amd import cue
from cuequivariance_amd.cuet import dense



def reference(e, w, x1, x2):
    """The product, one scaled matrix product per non-zero coefficient (ir_mul rows)."""
    stp = e.polynomial.operations[0][1]
    at = [o.segment_offsets() for o in stp.operands]
    columns = {}
    for p in stp.paths:
        sw, s1, s2, so = p.indices
        (d1, K), (d2, V), (d3, N) = stp.operands[1][s1], stp.operands[2][s2], stp.operands[3][so]
        W = w[0, at[0][sw]:at[0][sw] + K * V * N].view(K, V, N)
        for i, j, k in zip(*p.coefficients.nonzero()):
            a, b = x1[:, at[1][s1] + i * K:at[1][s1] + (i + 1) * K], x2[:, at[2][s2] + j * V:at[2][s2] + (j + 1) * V]
            t = float(p.coefficients[i, j, k]) * sum(b[:, v:v + 1] * (a @ W[:, v]) for v in range(V))
            key = at[3][so] + k * N
            columns[key] = columns[key] + t if key in columns else t
    return torch.cat([columns[k] for k in sorted(columns)], 1)


CASES = [
    ("64x0e+64x1o", "0e+1o", "64x0e+64x1o+64x1e", 40, torch.float32),
    ("96x0e+96x1o", "0e+1o+2e", "96x0e+96x1o+96x1e", 40, torch.bfloat16),
    ("16x0e+16x1o", "0e+1o", "16x0e+16x1o+16x1e", 13_100, torch.float32),  # (factors of the weight gradient through memory)
    ("96x0e+96x1o", "0e+1o", "96x0e+96x1o", 6_100, torch.bfloat16),
    ("48x0e+16x1o+32x2e", "2x0e+1x1o+5x2e", "32x0e+16x1o+48x2e", 40, torch.float32),
    ("48x0e+16x1o+32x2e", "2x0e+1x1o+5x2e", "32x0e+16x1o+48x2e", 40, torch.bfloat16),
    ("64x0e+64x1o", "16x0e+16x1o", "64x0e+64x1o+64x1e", 40, torch.bfloat16),  # (straight loops over the channels)
    ("32x0e+32x1o", "6x0e+6x1o+6x2e", "32x0e+32x1o+32x1e", 40, torch.bfloat16),
    ("32x0e+32x1o", "16x0e+16x1o", "32x0e+32x1o", 40, torch.float16),
]


@pytest.mark.gpu
@pytest.mark.parametrize("operand", ["x1", "x2", "g"])
@pytest.mark.parametrize("i1,i2,io,rows,dtype", CASES)
def test_an_infinite_component_reaches_what_it_is_coupled_to(device, i1, i2, io, rows, dtype, operand):
    from cuequivariance_amd import cuet

    i1, i2, io = (cue.Irreps("O3", i) for i in (i1, i2, io))
    m = cuet.FullyConnectedTensorProduct(i1, i2, io, layout=cue.ir_mul, internal_weights=False)
    e = cue.descriptors.fully_connected_tensor_product(i1, i2, io)
    g = torch.Generator().manual_seed(3)
    t = {n: torch.randn(*s, generator=g, dtype=torch.float64).to(dtype) for n, s in
         dict(w=(1, m.weight_numel), x1=(rows, i1.dim), x2=(rows, i2.dim), g=(rows, io.dim)).items()}
    irreps = {"x1": i1, "x2": i2, "g": io}[operand]
    first = irreps[0].mul * irreps[0].ir.dim  # the second block is 1o: its component 1, channel 0
    t[operand][rows // 2, first + irreps[1].mul] = float("inf")
    ref = {n: v.double().requires_grad_(n != "g") for n, v in t.items()}
    want = reference(e, ref["w"], ref["x1"], ref["x2"])
    want = [want, *torch.autograd.grad(want, [ref[n] for n in ("w", "x1", "x2")], ref["g"])]
    got_in = {n: v.to(device).requires_grad_(n != "g") for n, v in t.items()}
    out = m(got_in["x1"], got_in["x2"], got_in["w"])
    got = [out, *torch.autograd.grad(out, [got_in[n] for n in ("w", "x1", "x2")], got_in["g"])]
    spread = 0
    for name, a, b in zip(("out", "dw", "dx1", "dx2"), got, want):
        a, b = a.detach().cpu().double(), b.detach()
        keep = torch.isfinite(b)
        spread += int((~keep).sum())
        assert torch.isfinite(a[keep]).all(), (name, int((~torch.isfinite(a) & keep).sum()))
        if keep.any():  # (float32 sums of up to some 20 000 products; 2-byte results rounded once, formed factors once more)
            scale = b[keep].abs().max().item()
            assert (a[keep] - b[keep]).abs().max().item() <= {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}[dtype] * scale, name
    assert spread > 0


def test_the_straight_couplings_are_the_coefficients():
    """The rule that the straight kernels are compiled for covers the coefficients of every product it is applied to, and no more."""
    seen = set()
    e = cue.descriptors.fully_connected_tensor_product(*(cue.Irreps("O3", i) for i in ("0e+1o+1e", "0e+1o+2e", "0e+1o+1e")))
    for p in e.polynomial.operations[0][1].paths:
        d1, d2, d3 = p.coefficients.shape
        if (d1, d2, d3) in ((1, 1, 1), (1, 3, 3), (3, 3, 1), (3, 1, 3), (3, 3, 3), (3, 5, 3)):
            seen.add((d1, d2, d3))
            for i in range(d1):
                for j in range(d2):
                    for k in range(d3):
                        assert dense._couples(d1, d2, d3, i, j, k) == (p.coefficients[i, j, k] != 0), (d1, d2, d3, i, j, k)
    assert len(seen) == 6
