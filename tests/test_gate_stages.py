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
