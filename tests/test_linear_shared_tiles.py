"""Linear tiles that four wavefronts share (csrc/linear_flex.hip): contractions of fewer steps than wavefronts and of no multiple of
them, and the last number of rows whose tiles are shared with the first whose are not (4 column tiles: 512 tiles, 4 096 rows)."""

import pytest
import torch

from cuequivariance_amd import cue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("inner,outer,rows", [(16, 64, 1), (48, 32, 33), (80, 16, 65), (64, 64, 4096), (64, 64, 4097)])
def test_values_and_gradients(device, inner, outer, rows, dtype):
    from cuequivariance_amd import cuet

    # sums of up to 80 products of unit size, scaled to unit size: errors of some 2^-24 sqrt(80) in float; results rounded to 2^-9
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    i1, io = cue.Irreps("O3", f"{inner}x0e+{inner}x1o"), cue.Irreps("O3", f"{outer}x0e+{outer}x1o")
    m = cuet.Linear(i1, io, layout=cue.mul_ir, internal_weights=False)
    g = torch.Generator(device=device).manual_seed(rows)
    r = lambda *shape: torch.randn(*shape, device=device, generator=g).to(dtype)
    w, x, cot = r(1, m.weight_numel).requires_grad_(), r(rows, i1.dim).requires_grad_(), r(rows, io.dim)
    out = m(x, w)
    dx, = torch.autograd.grad(out, [x], cot)
    blocks = w.detach().double().reshape(2, inner, outer) / inner ** 0.5
    parts = lambda t, n: (t.double()[:, :n], t.double()[:, n:].reshape(rows, n, 3))
    x0, x1 = parts(x.detach(), inner)
    c0, c1 = parts(cot, outer)
    want = torch.cat([x0 @ blocks[0], torch.stack([x1[..., k] @ blocks[1] for k in range(3)], 2).reshape(rows, -1)], 1)
    want_dx = torch.cat([c0 @ blocks[0].T, torch.stack([c1[..., k] @ blocks[1].T for k in range(3)], 2).reshape(rows, -1)], 1)
    for got, ref in ((out.detach(), want), (dx, want_dx)):
        assert (got.double() - ref).abs().max().item() <= tol * ref.abs().max().item()
