"""The triangle update on squares whose side is no whole number of 16-byte pieces: the stages run on padded rows (mapped inside
the kernels, or copied in and out), and nothing of the padding may reach the caller's rows."""

import pytest
import torch

from oracle.triangle import triangle_multiplicative_update as oracle

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}


@pytest.mark.parametrize("all_weights", [True, False])
@pytest.mark.parametrize("batch,n,d,outgoing,dtype", [
    (1, 1, 32, True, torch.float32), (2, 3, 64, False, torch.bfloat16), (1, 7, 32, True, torch.float16),  # copied rows
    (2, 33, 64, True, torch.float32), (1, 66, 96, False, torch.bfloat16), (1, 21, 160, True, torch.float32),
    (1, 65, 128, True, torch.bfloat16), (1, 71, 64, False, torch.bfloat16), (3, 41, 128, False, torch.float16),  # mapped rows
    (1, 63, 64, True, torch.float16), (1, 391, 64, True, torch.bfloat16),
])
def test_ragged_squares_against_the_oracle(device, batch, n, d, outgoing, dtype, all_weights):
    from cuequivariance_amd import cuet

    g = torch.Generator().manual_seed(7)

    def r(*shape, scale=1.0, shift=0.0):
        return (torch.randn(*shape, generator=g, dtype=torch.float64) * scale + shift).to(dtype).double()

    p = dict(x=r(batch, n, n, d), mask=(torch.rand(batch, n, n, generator=g) < 0.9).double(), norm_in_weight=r(d, scale=0.1, shift=1.0),
             norm_in_bias=r(d, scale=0.1), p_in_weight=r(2 * d, d, scale=d ** -0.5), p_in_bias=r(2 * d, scale=0.1),
             g_in_weight=r(2 * d, d, scale=d ** -0.5), g_in_bias=r(2 * d, scale=0.1), norm_out_weight=r(d, scale=0.1, shift=1.0),
             norm_out_bias=r(d, scale=0.1), p_out_weight=r(d, d, scale=d ** -0.5), p_out_bias=r(d, scale=0.1), g_out_weight=r(d, d, scale=d ** -0.5),
             g_out_bias=r(d, scale=0.1))
    cot = r(batch, n, n, d)
    wanted = [k for k in p if k != "mask"] if all_weights else ["x"]
    direction = "outgoing" if outgoing else "incoming"
    ref_in = {k: v.clone().requires_grad_(k in wanted) for k, v in p.items()}
    ref = oracle(direction=direction, **ref_in)
    want = torch.autograd.grad(ref, [ref_in[k] for k in wanted], cot)
    got_in = {k: v.to(dtype).to(device).requires_grad_(k in wanted) for k, v in p.items()}
    out = cuet.triangle_multiplicative_update(direction=direction, **got_in)
    got = torch.autograd.grad(out, [got_in[k] for k in wanted], cot.to(dtype).to(device))
    for name, a, b in zip(["out", *wanted], [out, *got], [ref, *want]):
        assert a.dtype == dtype and a.shape == b.shape
        err = (a.detach().cpu().double() - b.detach()).abs().max().item()
        assert err <= TOL[dtype] * max(b.detach().abs().max().item(), 1e-3), (name, err, b.abs().max().item())
