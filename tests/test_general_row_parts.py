"""Kernels of the general generator (``codegen/general.py``) with an indexed output: one to sixteen wavefronts sharing the list of an
output row (``row_parts`` in ``csrc/cw_common.h``), against sums written out in torch - outputs with channels and scalar ones,
segments no path fills, lists that are empty, shorter than the parts, or hold nearly everything."""

import pytest
import torch

from cuequivariance_amd import _lib
from cuequivariance_amd.tables import U1dTables

TOL = {torch.float64: 1e-12, torch.float32: 2e-6}  # x largest value: sums of a few thousand products in order, or in parts

LISTS = {"sixteen parts": [100, 0, 33, 1, 700], "eight parts": [3, 40, 0, 9] * 50, "one part": [1, 0, 3] * 30, "two parts": [6, 2, 9] * 900}


def _run(device, tables, dtype, degrees, inputs, out_width, expect, ordered):
    from cuequivariance_amd.cuet.uniform_1d import Uniform1dPlan, run_plan

    Z, N = sum(degrees), len(degrees)
    g = torch.Generator().manual_seed(Z)
    rows = torch.repeat_interleave(torch.arange(N), torch.tensor(degrees))
    if not ordered:
        rows = rows[torch.randperm(Z, generator=g)]
    xs = [torch.randn(Z, n, generator=g, dtype=torch.float64).to(dtype).double() for n in inputs]
    want = torch.zeros(N, out_width, dtype=torch.float64).index_add(0, rows, expect(*xs))
    plan = Uniform1dPlan(tables, dtype, name="row_parts")
    B, I = _lib.BATCH_DIM_BATCHED, _lib.BATCH_DIM_INDEXED
    got = run_plan(plan, [B] * len(xs) + [I], [-1] * len(xs) + [0, N], Z, 1, [*(x.to(device, dtype) for x in xs), rows.int().to(device)])[0]
    assert plan.specialised(device)
    assert (got.cpu().double() - want).abs().max().item() <= TOL[dtype] * want.abs().max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("lists", LISTS)
def test_lists_of_an_output_with_channels(device, jit_on, lists, dtype):
    """s[] x[u] y[u] -> out[u]: eleven segments filled (more than meet in LDS at a time), one that nothing fills; 70 channels (two
    wavefronts' worth, the second with lanes to spare)."""
    E = 70
    paths = [(k % 3, (k + 1) % 2, k % 4, k if k < 5 else k + 1, 0.5 + k) for k in range(11)]
    tables = U1dTables.make(E, 3, 1, [0, 1, 1, 1], [4, 3, 2, 12], [0, 1, 2, -1], [4], [0, 1, 2, 3], [11], [0], [0],
                            [i for a, b, c, k, _ in paths for i in (c, a, b, k)], [p[4] for p in paths])

    def expect(s, x, y):
        out = torch.zeros(x.shape[0], 12, E, dtype=torch.float64)
        for a, b, c, k, f in paths:
            out[:, k] += f * x.reshape(-1, 3, E)[:, a] * y.reshape(-1, 2, E)[:, b] * s[:, c: c + 1]
        return out.reshape(-1, 12 * E)

    _run(device, tables, dtype, LISTS[lists], (4, 3 * E, 2 * E), 12 * E, expect, ordered=lists != "eight parts")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("lists", LISTS)
def test_lists_of_a_scalar_output(device, jit_on, lists, dtype):
    """x[u] gy[u] -> dw[] next to s[] gt[] -> dw[] (counted once, not once per channel), and a segment that nothing fills."""
    E = 48
    tables = U1dTables.make(E, 4, 1, [1, 1, 0, 0, 0], [2, 2, 2, 2, 3], [0, 1, 2, 3, -1], [3, 3], [0, 1, 4, 2, 3, 4], [3, 2], [0, 9], [0, 3],
                            [0, 0, 0, 1, 1, 2, 0, 1, 2, 0, 0, 0, 1, 0, 2], [2.0, -1.5, 0.5, 3.0, 0.25])

    def expect(x, gy, s, gt):
        x, gy = x.reshape(-1, 2, E), gy.reshape(-1, 2, E)
        first = 2.0 * (x[:, 0] * gy[:, 0]).sum(1) + 3.0 * s[:, 0] * gt[:, 0]
        last = -1.5 * (x[:, 1] * gy[:, 1]).sum(1) + 0.5 * (x[:, 0] * gy[:, 1]).sum(1) + 0.25 * s[:, 1] * gt[:, 0]
        return torch.stack([first, torch.zeros_like(first), last], 1)

    _run(device, tables, dtype, LISTS[lists], (2 * E, 2 * E, 2, 2), 3, expect, ordered=lists != "eight parts")
