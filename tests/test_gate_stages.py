"""The gate on products in memory (``cueq_gate_fwd``, ``cueq_gate_bwd``), and what goes through it: gated dual projections of operands
that are not 16-byte aligned."""

import pytest
import torch

from cuequivariance_amd import _lib

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}  # (float32 arithmetic, rounded once)


def test_the_entries_are_in_the_header():
    header = (_lib.LIB_PATH.parent.parent / "include" / "cueq_amd.h").read_text()
    for name in ("cueq_gate_fwd", "cueq_gate_bwd"):
        assert name in _lib.EXPORTED_SYMBOLS and f"int {name}(" in header and hasattr(_lib.load(), name)


@pytest.mark.parametrize("dtype", list(TOL))
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("aligned", [True, False])
def test_gated_projections(device, dtype, axis, aligned):
    from cuequivariance_amd.cuet import triangle as T

    g = torch.Generator().manual_seed(4)
    M, N, K = 70, 33, 32

    def r(*shape):
        t = torch.randn(*shape, generator=g, dtype=torch.float64)
        return t.to(dtype).double()

    def there(t, odd=False):  # odd: the same values from an address that is no multiple of 16 bytes
        flat = torch.empty(t.numel() + 1, dtype=dtype, device=device)
        view = flat[1:] if odd else flat[:-1]
        view.copy_(t.to(dtype).flatten())
        return view.view(t.shape)

    A1, A2, B1, B2, dout = r(M, K), r(M, K), r(N, K), r(N, K), r(M, N)
    n = M if axis == 0 else N
    b1, b2, mask = r(n), r(n), (torch.rand(n, generator=g) < 0.8).double()
    shape = (lambda t: t[:, None]) if axis == 0 else (lambda t: t[None, :])
    u, v = (A1 @ B1.T).requires_grad_(), (A2 @ B2.T).requires_grad_()
    ref = torch.sigmoid(u + shape(b1)) * (v + shape(b2)) * shape(mask)
    want = [ref, *torch.autograd.grad(ref, [u, v], dout)]
    args = [there(t, not aligned) for t in (A1, A2, B1, B2)]
    small = [there(b1), there(b2), axis, there(mask), axis]
    got = [T.dual_gate_fwd(*args, *small), *T.dual_gate_bwd(there(dout), *args, *small)]
    uf, vf = u.detach().float().to(device), v.detach().float().to(device)
    stage = [T.gate_fwd(uf, vf, *small, dtype), *T.gate_bwd(there(dout), uf, vf, *small)]
    for a, s, b in zip(got, stage, want):
        scale = b.detach().abs().max().item()
        assert a.dtype == s.dtype == dtype
        assert (a.cpu().double() - b.detach()).abs().max().item() <= TOL[dtype] * scale
        assert (s.cpu().double() - b.detach()).abs().max().item() <= TOL[dtype] * scale


@pytest.mark.parametrize("K,C", [(32, 32), (64, 96), (96, 32), (128, 256)])
@pytest.mark.parametrize("inputs,M", [(1, 4), (1, 36), (1, 128), (1, 132), (1, 3000), (2, 3), (2, 33), (2, 128), (2, 3001)])
def test_input_gradients_of_float32(device, inputs, M, K, C):
    """Down to the inputs in one kernel, 32 weight rows at a time (one, two, three and eight turns), 128 columns a block: with one input
    the cotangent and the gate gradients are (C, M), and the input's gradient may be added to what is there; with two they are (M, C)."""
    from cuequivariance_amd.cuet import triangle as T

    g = torch.Generator().manual_seed(M + K)
    r = lambda *shape: torch.randn(*shape, generator=g).double()
    X1, X2, W1, W2, b1, b2, before = r(M, K), r(M, K), r(C, K) / K ** 0.5, r(C, K) / K ** 0.5, r(C), r(C), r(M, K)
    mask, dout = (torch.rand(M, generator=g) < 0.8).double(), r(C, M)
    x1, x2 = X1.clone().requires_grad_(), X2.clone().requires_grad_()
    u, v = W1 @ x1.T, W2 @ (x1 if inputs == 1 else x2).T
    ref = torch.sigmoid(u + b1[:, None]) * (v + b2[:, None]) * mask
    dx1, du, dv, *dx2 = torch.autograd.grad(ref, [x1, u, v] + ([x2] if inputs == 2 else []), dout)
    f = lambda t: t.float().to(device)
    d = f(dout if inputs == 1 else dout.T.contiguous())
    for add in (False, True) if inputs == 1 else (False,):
        got = T.gate_bwd_input(d, inputs == 1, f(W1), f(W2), f(X1), f(X2) if inputs == 2 else None, f(b1), f(b2), f(mask), f(before) if add else None, True)
        want = [dx1 + before if add else dx1, dx2[0] if dx2 else None, *(t if inputs == 1 else t.T for t in (du, dv))]
        for a, b in zip(got, want):
            assert (a is None) == (b is None)
            # (float32 sums of up to 2 x 256 products)
            assert a is None or (a.cpu().double() - b).abs().max().item() <= 1e-5 * b.abs().max().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [32, 64, 96, 128])
@pytest.mark.parametrize("M", [1, 31, 33, 8191, 65_569])
def test_two_inputs_with_as_many_weight_rows_as_columns(device, M, K, dtype):
    """The output stage in 2-byte types: parts of a tile of 32 rows, and one wavefront with a second tile (65 569 rows are 2 050 tiles for
    2 048 wavefronts); with and without gate gradients, mask and biases."""
    from cuequivariance_amd.cuet import triangle as T

    g = torch.Generator().manual_seed(M + K)
    r = lambda *shape: torch.randn(*shape, generator=g).to(dtype).float().to(device)
    X1, X2, W1, W2, b1, b2, dout = r(M, K), r(M, K), r(K, K) / 8, r(K, K) / 8, r(K), r(K), r(M, K)
    mask = (torch.rand(M, generator=g) < 0.8).float().to(device)
    f = lambda t: t.to(dtype)
    for plain in (False, True):
        x1, x2 = X1.clone().requires_grad_(), X2.clone().requires_grad_()
        u, v = x1 @ W1.T + (0 if plain else b1), x2 @ W2.T + (0 if plain else b2)
        want = torch.autograd.grad(torch.sigmoid(u) * v * (1 if plain else mask[:, None]), [x1, x2, u, v], dout)
        few = (None, None, None) if plain else (f(b1), f(b2), f(mask))
        got = T.gate_bwd_input(f(dout), False, f(W1), f(W2), f(X1), f(X2), *few, None, not plain)
        for a, b in zip(got, want):
            # (the gate gradients are rounded once and so is the result: with unit roundoff e, e (sum |du w| / max |dx| + 1) of the largest
            # value, the sum of K random products about twice the largest result)
            assert (plain and a is None) or (a.float() - b).abs().max().item() <= TOL[dtype] * b.abs().max().item()
