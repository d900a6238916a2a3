"""Linear tiles whose rows are staged through LDS (``flex_stage_kernel`` in ``csrc/linear_flex.hip``): one to five column tiles of a block
(the workgroup's four, two and one beside each other), contractions that end inside a group of four steps, sums over input
blocks, up to seven components, ragged rows, and the taller slabs of many rows in ir_mul."""

import pytest
import torch

from cuequivariance_amd import cue

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def tables_alone(monkeypatch):
    """No row-streaming or tiled launches, whatever the number of rows (rows in mul_ir have theirs from 55 000 rows on, past all cases here)."""
    from cuequivariance_amd.cuet import dense

    monkeypatch.setattr(dense, "_rows_launches", lambda mod, es: None)


def _check(device, irreps_in, irreps_out, rows, dtype, layout):
    from cuequivariance_amd import cuet

    # sums of up to 320 products of unit size, scaled to unit size: errors of some 2^-24 sqrt(320) in float; results rounded to 2^-9, 2^-12
    tol = {torch.float32: 1e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}[dtype]
    i1, io = cue.Irreps("O3", irreps_in), cue.Irreps("O3", irreps_out)
    m = cuet.Linear(i1, io, layout=layout, internal_weights=False, method="fused_tp")
    g = torch.Generator(device=device).manual_seed(rows)
    r = lambda *shape: torch.randn(*shape, device=device, generator=g).to(dtype)
    w, x, cot = r(1, m.weight_numel), r(rows, i1.dim).requires_grad_(), r(rows, io.dim)
    out = m(x, w)
    dx, = torch.autograd.grad(out, [x], cot)

    def blocks(t, irreps):  # per irrep copy block: (rows, mul, dim) in 64 bits
        parts, at = [], 0
        for mul, ir in irreps:
            b = t[:, at: at + mul * ir.dim].double()
            parts.append(b.reshape(rows, mul, ir.dim) if layout == cue.mul_ir else b.reshape(rows, ir.dim, mul).transpose(1, 2))
            at += mul * ir.dim
        return parts

    xs, cs = blocks(x.detach(), i1), blocks(cot, io)
    want, want_dx, at = [torch.zeros_like(c) for c in cs], [torch.zeros_like(b) for b in xs], 0
    pairs = [(a, b) for a, (_, ia) in enumerate(i1) for b, (_, ib) in enumerate(io) if ia == ib]
    fan = {b: sum(i1[a].mul for a, bb in pairs if bb == b) for _, b in pairs}
    for a, b in pairs:
        block = w[0, at: at + i1[a].mul * io[b].mul].double().reshape(i1[a].mul, io[b].mul) / fan[b] ** 0.5
        at += block.numel()
        want[b] += torch.einsum("zud,uv->zvd", xs[a].cpu(), block.cpu()).to(device)
        want_dx[a] += torch.einsum("zvd,uv->zud", cs[b].cpu(), block.cpu()).to(device)
    for got, ref in ((out.detach(), (want, io)), (dx, (want_dx, i1))):
        for p, q in zip(blocks(got, ref[1]), ref[0]):
            assert (p - q).abs().max().item() <= tol * q.abs().max().item()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", [cue.mul_ir, cue.ir_mul])
@pytest.mark.parametrize("irreps_in,irreps_out,rows", [
    ("48x0e+16x1o+80x2e+16x3o", "160x0e+96x1o+64x2e+16x3o", 2081),      # 5, 3, 2 and 1 column tiles; one to five steps of 2-byte elements
    ("16x0e+160x0e+144x1o+32x1o", "128x0e+48x1o+32x1o", 3000),          # sums over input blocks; a tile that is half empty
    ("32x0e+32x1o+32x2e+32x3o", "32x0e+32x1o+32x2e+32x3o", 16384 + 1),  # one column tile; one row in the last slab
])
def test_against_64_bits(device, irreps_in, irreps_out, rows, layout, dtype):
    _check(device, irreps_in, irreps_out, rows, dtype, layout)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("irreps_in,irreps_out,rows", [
    ("144x0e+48x1o", "144x0e+48x1o", 40_001),  # five and two column tiles of a block: groups of four, two and one
    ("80x0e+80x1o", "96x0e+32x1o", 60_007),    # three and one
])
def test_taller_slabs(device, irreps_in, irreps_out, rows, dtype):
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    for irreps in (irreps_in, irreps_out):  # (four row tiles a wavefront from so many workgroups of one on)
        tiles = sum(-(-mul // 32) * ir.dim for mul, ir in cue.Irreps("O3", irreps))
        assert -(-rows // 128) * tiles >= (9 if dtype == torch.float32 else 4) * cus
    _check(device, irreps_in, irreps_out, rows, dtype, cue.ir_mul)
