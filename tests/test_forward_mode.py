"""Forward-mode differentiation is not offered: a call with a tangent is refused on every path, never computed without it."""

import pytest
import torch
import torch.autograd.forward_ad as forward_ad

from cuequivariance_amd import cue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["linear", "fully", "general", "channelwise", "triangle"])
@pytest.mark.parametrize("which", [0, 1])
def test_a_tangent_is_refused(device, kind, which):
    from cuequivariance_amd import cuet

    irreps = cue.Irreps("O3", "32x0e+32x1o")
    r = lambda *shape: torch.randn(*shape, device=device)
    options = dict(layout=cue.ir_mul, internal_weights=False)
    if kind == "linear":
        m = cuet.Linear(irreps, irreps, **options)
        args = [r(5, irreps.dim), r(1, m.weight_numel)]
    elif kind in ("fully", "general"):
        second = cue.Irreps("O3", "0e+1o" if kind == "fully" else "16x0e+16x1o")
        m = cuet.FullyConnectedTensorProduct(irreps, second, irreps, **options)
        args = [r(5, irreps.dim), r(5, second.dim), r(1, m.weight_numel)]
    elif kind == "channelwise":
        second = cue.Irreps("O3", "0e+1o+2e")
        m = cuet.ChannelWiseTensorProduct(cue.Irreps("O3", "32x0e+32x1o+32x2e"), second, "0e+1o+2e", shared_weights=False, **options)
        args = [r(5, m.irreps_in1.dim), r(5, second.dim), r(5, m.weight_numel)]
    else:
        weights = dict(norm_in_weight=r(64), norm_in_bias=r(64), p_in_weight=r(128, 64), g_in_weight=r(128, 64), norm_out_weight=r(64), norm_out_bias=r(64),
                       p_out_weight=r(64, 64), g_out_weight=r(64, 64))
        m = lambda x, p: cuet.triangle_multiplicative_update(x, direction="outgoing", **dict(weights, p_in_weight=p))
        args = [r(1, 16, 16, 64), weights["p_in_weight"]]
    with torch.no_grad():
        m(*args)
    with forward_ad.dual_level():
        args[which] = forward_ad.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises((RuntimeError, NotImplementedError)):
            m(*args)
