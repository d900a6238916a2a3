"""The first call of a module may be one that is captured into a HIP graph, where there are launches whose tables are kernel arguments:
``mul_ir`` Linears of 32, 64, 96 or 128 channels and the fully connected products with generated kernels, of few rows or many."""

import pytest
import torch

from cuequivariance_amd import cue

pytestmark = pytest.mark.gpu


def linear(device, mul, rows, dtype):
    from cuequivariance_amd import cuet

    irreps = cue.Irreps("O3", f"{mul}x0e+{mul}x1o")
    m = cuet.Linear(irreps, irreps, layout=cue.mul_ir, internal_weights=False)
    shapes = [(rows, irreps.dim), (1, m.weight_numel)]
    return m, shapes, irreps.dim


def fully(device, mul, rows, dtype):
    from cuequivariance_amd import cuet

    irreps, second = cue.Irreps("O3", f"{mul}x0e+{mul}x1o"), cue.Irreps("O3", "0e+1o+2e")
    m = cuet.FullyConnectedTensorProduct(irreps, second, irreps, layout=cue.mul_ir, internal_weights=False)
    return m, [(rows, irreps.dim), (rows, second.dim), (1, m.weight_numel)], irreps.dim


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("make,mul,rows,dtype", [(linear, 128, 37, torch.float32), (linear, 64, 300, torch.bfloat16), (linear, 128, 25_000, torch.float32),
                                                 (fully, 64, 300, torch.float32), (fully, 64, 300, torch.bfloat16)])
def test_capture_without_a_call_before(device, jit_on, make, mul, rows, dtype, train):
    g = torch.Generator().manual_seed(rows)

    def setup():
        m, shapes, width = make(device, mul, rows, dtype)
        return m, [torch.empty(*s, dtype=dtype, device=device).requires_grad_(train) for s in shapes], torch.empty(rows, width, dtype=dtype, device=device)

    def step(m, args, cot):
        out = m(*args)
        return [out, *torch.autograd.grad(out, args, cot)] if train else [out]

    def fill(tensors):
        with torch.no_grad():
            for t in tensors:
                t.copy_(torch.randn(*t.shape, generator=g))

    other = setup()  # (another module of the same kind: the library, not the module, has run before)
    fill([*other[1], other[2]])
    step(*other)
    torch.cuda.synchronize()
    m, args, cot = setup()
    fill([*args, cot])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        results = step(m, args, cot)
    for _ in range(3):
        fill([*args, cot])
        graph.replay()
        torch.cuda.synchronize()
        got = [r.clone() for r in results]
        want = step(*(other[0], args, cot))
        torch.cuda.synchronize()
        for a, b in zip(got, want):  # (the eager call may take other kernels: float32 sums in another order, 2-byte results rounded once)
            assert (a - b).abs().max().item() <= (1e-5 if dtype == torch.float32 else 1e-2) * b.abs().max().item()
