"""The division of 3-vectors by their length in front of the spherical harmonics (``csrc/row_scale.hip``), with its first, second and
third derivatives, against ``torch.nn.functional.normalize`` in 64 bits: vectors of ordinary length, shorter than its eps, zero,
of every remainder of a wavefront."""

import pytest
import torch

from cuequivariance_amd import _lib

pytestmark = pytest.mark.gpu
# float32: a handful of roundings (6e-8 each) of terms that cancel to a tenth or so of themselves in the second derivative
TOL = {torch.float64: 1e-13, torch.float32: 4e-6}


def _derivatives(normalize, x, g, v, u):
    x, g, v = (t.clone().requires_grad_(True) for t in (x, g, v))
    y = normalize(x)
    (dx,) = torch.autograd.grad(y, x, g, create_graph=True)
    first = torch.autograd.grad(dx, [g, x], v, create_graph=True)
    third = torch.autograd.grad(first[1], [x, g, v], u, retain_graph=True)
    plain = torch.autograd.grad(dx, [g, x], v.detach())  # (without a graph: the kernel)
    return [y, dx, *plain, *first, *third]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 1000])
def test_against_pytorch_in_64_bits(device, rows, dtype):
    g = torch.Generator().manual_seed(rows)
    x, *rest = (torch.randn(rows, 3, generator=g, dtype=torch.float64).to(dtype) for _ in range(4))
    want = _derivatives(lambda t: torch.nn.functional.normalize(t, dim=1), x.double(), *[t.double() for t in rest])
    x = x.to(device).t().contiguous().t()  # (rows that are not contiguous)
    got = _derivatives(_lib.host().normalize, x, *[t.to(device) for t in rest])
    for k, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == dtype
        err = (a.cpu().double() - b).norm(dim=1) / b.norm(dim=1).clamp(min=1e-3 * b.norm(dim=1).max().item())
        assert err.max().item() <= (10 if k > 5 else 1) * 8 * TOL[dtype], (k, err.max().item())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_short_zero_and_odd_vectors(device, dtype):
    """Below eps the divisor is a constant: finite derivatives (PyTorch's second derivative of a zero vector is 0 / 0); NaN and
    infinity come out where PyTorch has them."""
    inf, nan = float("inf"), float("nan")
    x = torch.tensor([[0.0, 0, 0], [1e-14, 0, -2e-14], [1e-10, 1e-10, 0], [1, 2, 3], [nan, 1, 2], [inf, 1, 2], [1e12, 0, 1e12]], dtype=dtype, device=device)
    g = torch.randn(7, 3, generator=torch.Generator().manual_seed(0)).to(device, dtype)
    out = []
    for normalize in (_lib.host().normalize, lambda t: torch.nn.functional.normalize(t, dim=1)):
        a, b = x.clone().requires_grad_(True), g.clone().requires_grad_(True)
        y = normalize(a)
        (dx,) = torch.autograd.grad(y, a, b, create_graph=True)
        out.append([y, dx, *torch.autograd.grad(dx, [b, a], torch.ones_like(g))])
    for k, (got, want) in enumerate(zip(*out)):
        first = 1 if k >= 2 else 0
        # (rounding errors of a row's terms, whose size is at most a few times the largest |v| |g| / |x|^k of the row: not of each entry, which
        # may cancel to nothing, and not of the other rows, 1e10 times shorter or longer)
        scale = torch.ones_like(g)[first:4].norm(dim=1) * g[first:4].norm(dim=1) if k == 3 else want[first:4].norm(dim=1).clamp(min=1.0)
        bound = (1e-5 if dtype == torch.float32 else 1e-12) * scale / x[first:4].norm(dim=1).clamp(min=1e-12) ** (2 if k == 3 else 0)
        assert ((got - want)[first:4].norm(dim=1) <= bound).all(), k
        assert got[0].isfinite().all()
        assert torch.equal(got[6].isfinite(), want[6].isfinite())
    for k in (0, 1, 2):
        assert torch.equal(out[0][k][4:].isnan(), out[1][k][4:].isnan())


@pytest.mark.parametrize("graph", [False, True])
def test_second_derivative_keeps_nan(device, graph):
    """What no length divides has no second derivative either: NaN, with a graph (PyTorch's operations) and without (the kernel)."""
    x = torch.tensor([[float("nan"), 1, 2], [float("inf"), 1, 2], [1, 2, 3]], device=device, requires_grad=True)
    g = torch.ones_like(x).requires_grad_()
    (dx,) = torch.autograd.grad(_lib.host().normalize(x), x, g, create_graph=True)
    for second in torch.autograd.grad(dx, [g, x], torch.ones_like(x), create_graph=graph):
        assert second[:2].isnan().all() and second[2].isfinite().all()


def test_calls_that_are_not_plain_are_left_to_pytorch(device):
    normalize = _lib.host().normalize
    x = torch.randn(4, 3, device=device)
    assert normalize(x) is not None and normalize(x[:0]).shape == (0, 3)
    assert normalize(x.cpu()) is None and normalize(x.half()) is None and normalize(x[:, :2]) is None and normalize(x[0]) is None
    seen = []
    torch.func.vmap(lambda t: (seen.append(normalize(t)), t)[1])(x.reshape(2, 2, 3))
    assert seen == [None]
