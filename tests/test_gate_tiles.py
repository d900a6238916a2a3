"""How the gate kernels with resident weights deal out their tiles - over the CUs first and, for few of them, over the weight rows as
well (four or eight parts of 64-row tiles up to 8 192 rows, two or four of 32-row tiles) - must not show in a result: every row has the
bits it has among 70 008 rows, whose tiles fill the device.  (Against float64: tests/test_triangle.py, rows of padded
squares, which take the same parts: tests/test_triangle_padded.py.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu

MANY = 70_008


@pytest.mark.parametrize("M", [4096, 4104, 8184, 16_384, 16_456, 33_000])
@pytest.mark.parametrize("K,C", [(128, 256), (64, 96), (32, 32)])
def test_rows_do_not_depend_on_how_tiles_are_dealt_out(device, M, K, C):
    from cuequivariance_amd.cuet import triangle as T

    g = torch.Generator(device=device).manual_seed(M + K)
    rn = lambda *shape: torch.randn(*shape, device=device, generator=g).bfloat16()
    x, x2, gamma, beta, b1, b2 = rn(MANY, K), rn(MANY, K), rn(K), rn(K), rn(C), rn(C)
    W1, W2, mask, d, dr = rn(C, K), rn(C, K), rn(MANY), rn(C, MANY), rn(MANY, C)

    def run(m):
        xs, x2s, ms = x[:m], x2[:m], mask[:m]
        out, xh, mean, rstd = T.ln_dual_gate_fwd(xs, gamma, beta, 1e-5, W1, W2, b1, b2, ms)
        one = T.dual_gate_fwd(W1, W2, xs, None, b1, b2, 0, ms, 1)
        rows = T.dual_gate_fwd(xs, x2s, W1, W2, b1, b2, 1, ms, 0)
        dx, _, du, dv = T.gate_bwd_input(d[:, :m].contiguous(), True, W1, W2, xs, None, b1, b2, ms, want_gate_grads=True)
        dx1, dx2, du2, dv2 = T.gate_bwd_input(dr[:m], False, W1, W2, xs, x2s, b1, b2, ms, want_gate_grads=True)
        return (out, one, du, dv), (xh, mean, rstd, rows, dx, dx1, dx2, du2, dv2)

    (cols, rows), (cols_of_many, rows_of_many) = run(M), run(MANY)
    for a, b in zip(cols, cols_of_many):
        assert torch.equal(a, b[:, :M])
    for a, b in zip(rows, rows_of_many):
        assert torch.equal(a, b[:M])
