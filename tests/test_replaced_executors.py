"""The direct native way of the modules is for the executor they were built with: a replaced or wrapped one is called, and hooks on the
executor (profilers, operation counters) see every call."""

import pytest
import torch

from cuequivariance_amd import cue

pytestmark = pytest.mark.gpu


class Counting(torch.nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner, self.calls = inner, 0

    def forward(self, *args, **kwargs):
        self.calls += 1
        return self.inner(*args, **kwargs)


def case(kind, device):
    from cuequivariance_amd import cuet

    irreps, g = cue.Irreps("O3", "32x0e+32x1o"), torch.Generator().manual_seed(1)
    r = lambda *shape: torch.randn(*shape, generator=g).to(device)
    layout = cue.mul_ir if kind.endswith("mul_ir") else cue.ir_mul
    kind = kind.replace("_mul_ir", "")
    options = dict(layout=layout, internal_weights=False)
    if kind == "linear":
        m = cuet.Linear(irreps, irreps, **options)
        return m, [r(9, irreps.dim), r(1, m.weight_numel)]
    if kind in ("fully", "general"):
        second = cue.Irreps("O3", "0e+1o" if kind == "fully" else "16x0e+16x1o")
        m = cuet.FullyConnectedTensorProduct(irreps, second, irreps, **options)
        return m, [r(9, irreps.dim), r(9, second.dim), r(1, m.weight_numel)]
    if kind == "channelwise":
        m = cuet.ChannelWiseTensorProduct(cue.Irreps("O3", "32x0e+32x1o+32x2e"), cue.Irreps("O3", "0e+1o+2e"), "0e+1o+2e", shared_weights=False, **options)
        return m, [r(9, m.irreps_in1.dim), r(9, m.irreps_in2.dim), r(9, m.weight_numel)]
    if kind == "channelwise_sh":
        m = cuet.ChannelWiseSphericalTensorProduct(cue.Irreps("O3", "32x0e+32x1o+32x2e"), [0, 1, 2], "0e+1o+2e", shared_weights=False, **options)
        return m, [r(9, m.irreps_in1.dim), r(9, 3), r(9, m.weight_numel)]
    if kind == "contraction":
        m = cuet.SymmetricContraction(irreps, cue.Irreps("O3", "32x0e"), 2, 3, layout=layout).to(device)
        return m, [r(9, irreps.dim), torch.randint(0, 3, (9,), generator=g, dtype=torch.int32).to(device)]
    return cuet.SphericalHarmonics([0, 1, 2], normalize=False), [r(9, 3)]


KINDS = ["linear", "linear_mul_ir", "fully", "fully_mul_ir", "general", "general_mul_ir", "channelwise", "channelwise_mul_ir", "channelwise_sh",
         "contraction", "contraction_mul_ir", "harmonics"]


def executors(m):
    """The children that run the product: one of them is called, whichever serves the layout and the type."""
    return [name for name in ("f", "f_rows") if m._modules.get(name) is not None]


def same(a, b):
    assert (a - b).abs().max().item() <= 1e-5 * b.abs().max().item()  # (float32 sums, possibly by another kernel)


@pytest.mark.parametrize("kind", KINDS)
def test_a_wrapped_executor_is_called(device, kind):
    m, args = case(kind, device)
    want = m(*args)
    wrapped = []
    for name in executors(m):
        setattr(m, name, Counting(getattr(m, name)))
        wrapped.append(getattr(m, name))
    same(m(*args), want)
    assert sum(w.calls for w in wrapped) == 1


@pytest.mark.parametrize("kind", KINDS)
def test_a_compiled_executor(device, kind):
    m, args = case(kind, device)
    want = m(*args)
    for name in executors(m):
        setattr(m, name, torch.compile(getattr(m, name), backend="eager"))
    same(m(*args), want)


@pytest.mark.parametrize("depth", ["f", "f.m"])
@pytest.mark.parametrize("kind", KINDS)
def test_hooks_are_called(device, kind, depth):
    m, args = case(kind, device)
    want, seen = m(*args), []
    handles = []
    for name in executors(m):
        child = getattr(m, name) if depth == "f" else getattr(m, name).m
        handles += [child.register_forward_pre_hook(lambda *_: seen.append("before")), child.register_forward_hook(lambda *_: seen.append("after"))]
    same(m(*args), want)
    assert seen == ["before", "after"]
    for h in handles:
        h.remove()
    same(m(*args), want)
    assert len(seen) == 2


@pytest.mark.parametrize("kind", KINDS)
def test_global_hooks_and_replaced_forwards(device, kind):
    m, args = case(kind, device)
    want, seen = m(*args), []
    children = [getattr(m, name) for name in executors(m)]
    handle = torch.nn.modules.module.register_module_forward_hook(lambda module, *_: seen.append(module) if module in children else None)
    same(m(*args), want)
    handle.remove()
    assert len(seen) == 1
    for child in children:
        inner = child.forward
        child.forward = lambda *a, _inner=inner, **k: (seen.append("replaced"), _inner(*a, **k))[1]
    same(m(*args), want)
    assert seen[1:] == ["replaced"]
