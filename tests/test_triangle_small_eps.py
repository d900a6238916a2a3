"""The triangle update with ``eps = 0`` on squares whose side is no whole number of 16-byte pieces: what the padding holds must not make
the caller's rows or gradients infinite or NaN (a row of zeros has no deviation to divide by)."""

import pytest
import torch

from oracle.triangle import triangle_multiplicative_update as oracle

pytestmark = pytest.mark.gpu
# (the tolerances of the same squares with the default eps; without eps the reciprocal deviations are those of the rows themselves, of
# order one for these inputs, and nothing is amplified)
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("batch,n,d,outgoing,dtype", [
    (1, 9, 32, True, torch.float32), (1, 9, 32, False, torch.float32), (2, 13, 64, True, torch.bfloat16), (1, 21, 96, False, torch.float16),
    (1, 5, 288, False, torch.float32),  # copied rows; d > 256 with a transposed copy
    (1, 67, 64, True, torch.bfloat16), (1, 67, 64, False, torch.float16), (1, 71, 128, True, torch.float16), (1, 71, 128, False, torch.bfloat16),  # mapped
])
def test_no_eps_on_ragged_squares(device, batch, n, d, outgoing, dtype, masked):
    from cuequivariance_amd import cuet

    g = torch.Generator().manual_seed(5)

    def r(*shape, scale=1.0, shift=0.0):
        return (torch.randn(*shape, generator=g, dtype=torch.float64) * scale + shift).to(dtype).double()

    p = dict(x=r(batch, n, n, d), norm_in_weight=r(d, scale=0.1, shift=1.0), p_in_weight=r(2 * d, d, scale=d ** -0.5),
             g_in_weight=r(2 * d, d, scale=d ** -0.5), norm_out_weight=r(d, scale=0.1, shift=1.0), norm_out_bias=r(d, scale=0.1),
             p_out_weight=r(d, d, scale=d ** -0.5), g_out_weight=r(d, d, scale=d ** -0.5))
    if masked:
        p["mask"] = (torch.rand(batch, n, n, generator=g) < 0.9).double()
    cot = r(batch, n, n, d)
    wanted = [k for k in p if k != "mask"]
    options = dict(direction="outgoing" if outgoing else "incoming", eps=0.0)
    ref_in = {k: v.clone().requires_grad_(k in wanted) for k, v in p.items()}
    ref = oracle(**options, **ref_in)
    want = torch.autograd.grad(ref, [ref_in[k] for k in wanted], cot)
    got_in = {k: v.to(dtype).to(device).requires_grad_(k in wanted) for k, v in p.items()}
    out = cuet.triangle_multiplicative_update(**options, **got_in)
    got = torch.autograd.grad(out, [got_in[k] for k in wanted], cot.to(dtype).to(device))
    for name, a, b in zip(["out", *wanted], [out, *got], [ref, *want]):
        err = (a.detach().cpu().double() - b.detach()).abs().max().item()
        assert err <= TOL[dtype] * max(b.detach().abs().max().item(), 1e-3), (name, err, b.abs().max().item())


@pytest.mark.parametrize("n,d,outgoing,dtype", [(9, 32, True, torch.float32), (13, 64, False, torch.bfloat16), (67, 64, False, torch.bfloat16),
                                                (71, 128, True, torch.float16)])
@pytest.mark.parametrize("row,column", [(-1, -1), (2, -1), (-1, 3), (4, 5)])
def test_an_infinite_value_stays_in_its_rows(device, n, d, outgoing, dtype, row, column):
    """Padding repeats the last row and column: what is infinite there must not reach rows that it does not reach without padding."""
    from cuequivariance_amd import cuet

    g = torch.Generator().manual_seed(6)
    r = lambda *shape, scale=1.0: (torch.randn(*shape, generator=g, dtype=torch.float64) * scale).to(dtype).double()
    p = dict(x=r(1, n, n, d), p_in_weight=r(2 * d, d, scale=d ** -0.5), g_in_weight=r(2 * d, d, scale=d ** -0.5), p_out_weight=r(d, d, scale=d ** -0.5),
             g_out_weight=r(d, d, scale=d ** -0.5), p_in_bias=r(2 * d), g_in_bias=r(2 * d))
    p["x"][0, row, column, 7] = float("inf")
    options = dict(direction="outgoing" if outgoing else "incoming")
    want = oracle(**options, **p)
    got = cuet.triangle_multiplicative_update(**options, **{k: v.to(dtype).to(device) for k, v in p.items()}).cpu().double()
    keep = torch.isfinite(want)
    assert keep.any() and not keep.all() and torch.equal(torch.isfinite(got), keep)
    assert (got[keep] - want[keep]).abs().max().item() <= TOL[dtype] * want[keep].abs().max().item()
