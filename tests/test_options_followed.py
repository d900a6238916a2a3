"""``CUEQ_DETERMINISTIC`` is looked at by every launch of the uniform-1d operator, also by a backward whose forward has seen another
value."""

import pytest
import torch

from cuequivariance_amd import _lib, cue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("second", [False, True])
def test_a_change_between_forward_and_backward(device, monkeypatch, second):
    from cuequivariance_amd import cuet

    monkeypatch.setenv("CUEQ_DETERMINISTIC", "0")
    m = cuet.ChannelWiseTensorProduct(cue.Irreps("O3", "32x0e+32x1o"), cue.Irreps("O3", "0e+1o"), "0e+1o", layout=cue.ir_mul, shared_weights=False,
                                      internal_weights=False)
    g = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g).to(device).requires_grad_(True)
    x1, x2, w = r(5, m.irreps_in1.dim), r(40, m.irreps_in2.dim), r(40, m.weight_numel)
    senders = torch.randint(0, 5, (40,), generator=g, dtype=torch.int32).to(device)
    out = m(x1, x2, w, indices_1=senders)
    assert _lib.get_option("deterministic") == 0
    if second:
        first = torch.autograd.grad(out.square().sum(), [x1, x2], create_graph=True)
        out = first[0].square().sum() + first[1].square().sum()
    monkeypatch.setenv("CUEQ_DETERMINISTIC", "1")
    a = torch.autograd.grad(out.sum(), [x1, w], retain_graph=True)
    assert _lib.get_option("deterministic") == 1
    b = torch.autograd.grad(out.sum(), [x1, w])
    assert all(torch.equal(p, q) for p, q in zip(a, b))
    monkeypatch.setenv("CUEQ_DETERMINISTIC", "0")
    m(x1, x2, w, indices_1=senders)
    assert _lib.get_option("deterministic") == 0
