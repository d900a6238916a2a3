"""Indexed channel-wise products where the rows are few and the lists uneven: one, four and eight wavefronts sharing the list of
an output row (``fwd_parts`` in ``csrc/cw_common.h``), wavefronts of the backward with one batch row each, and lists that are
empty, shorter than the parts, or hold nearly everything."""

import pytest
import torch

from cuequivariance_amd import cue

TOL = {torch.float64: 1e-12, torch.float32: 1e-5}  # x largest value, sums of at most 700 terms
DESCRIPTORS = {"c32_l2": ("32x0e+32x1o+32x2e", "0e+1o+2e", "0e+1o+2e"), "c128_l3": ("128x0e+128x1o+128x2e+128x3o", "0e+1o+2e+3o", "0e+1o+2e+3o"),
               "c16_l1": ("16x0e+16x1o", "0e+1o", "0e+1o"), "c24_l1": ("24x0e+24x1o", "0e+1o", "0e+1o"), "c5_l1": ("5x0e+5x1o", "0e+1o", "0e+1o")}


def _case(device, name, degrees, dtype, layout, ordered=True):
    from cuequivariance_amd import cuet
    from oracle.naive import naive_segmented_polynomial, spec_from_polynomial
    from tests.test_mul_ir_addressing import assert_close, to_mul_ir

    ir1, ir2, filt = DESCRIPTORS[name]
    ir1, ir2 = cue.Irreps("O3", ir1), cue.Irreps("O3", ir2)
    m = cuet.ChannelWiseTensorProduct(ir1, ir2, filt, layout=layout, shared_weights=False)
    into1, into3 = [(lambda x, i=i: to_mul_ir(x, i)) if layout == cue.mul_ir else (lambda x: x) for i in (ir1, m.irreps_out)]
    g = torch.Generator().manual_seed(len(degrees))
    N, Z = len(degrees), sum(degrees)
    receivers = torch.repeat_interleave(torch.arange(N, dtype=torch.int32), torch.tensor(degrees))
    if not ordered:
        receivers = receivers[torch.randperm(Z, generator=g)]
    senders = torch.randint(0, N, (Z,), generator=g, dtype=torch.int32)
    w, x1, x2, cot = (torch.randn(*s, dtype=torch.float64, generator=g).to(dtype).double()
                      for s in ((Z, m.weight_numel), (N, ir1.dim), (Z, ir2.dim), (N, m.irreps_out.dim)))
    a = [t.clone().requires_grad_(True) for t in (w, x1, x2)]
    ref = naive_segmented_polynomial(spec_from_polynomial(m.f._polynomial_orig), a, {1: senders}, {0: N}, {0: receivers})[0]
    ref_grads = torch.autograd.grad(ref, a, cot)
    b = [t.to(device, dtype).requires_grad_(True) for t in (w, into1(x1), x2)]
    out = m(b[1], b[2], b[0], indices_1=senders.to(device), indices_out=receivers.to(device), size_out=N)
    grads = torch.autograd.grad(out, b, into3(cot).to(device, dtype))
    assert m.f.m._plan(dtype).specialised(device)
    for what, got, want in zip(("out", "dw", "dx1", "dx2"), (out, *grads), (into3(ref), ref_grads[0], into1(ref_grads[1]), ref_grads[2])):
        assert_close(got, want, TOL[dtype], what)


# (rows, lists): eight parts, four parts, one part - the last by many rows, or by lists too short to share
LISTS = {"one row": [41], "eight parts": [0, 300, 1, 7, 8, 9, 64], "four parts": [3, 0, 17, 9, 40] * 20, "short lists": [2, 0, 1, 3] * 9,
         "many rows": [9] * 1100, "one batch row": [0, 1, 0]}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("layout", [cue.mul_ir, cue.ir_mul])
@pytest.mark.parametrize("lists", LISTS)
def test_lists_shared_by_wavefronts_32_channels(device, lists, layout, dtype):
    _case(device, "c32_l2", LISTS[lists], dtype, layout, ordered=lists != "four parts")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("lists", ["one row", "eight parts", "four parts"])
def test_lists_shared_by_wavefronts_128_channels(device, lists, dtype):
    _case(device, "c128_l3", LISTS[lists], dtype, cue.mul_ir, ordered=lists != "four parts")


@pytest.mark.gpu
@pytest.mark.parametrize("name,dtype,layout", [("c16_l1", torch.float32, cue.mul_ir), ("c24_l1", torch.float32, cue.ir_mul), ("c24_l1", torch.float64, cue.mul_ir),
                                               ("c5_l1", torch.float32, cue.mul_ir)])
def test_lists_shared_by_wavefronts_few_channels(device, jit_on, name, dtype, layout):
    for lists in ("one row", "eight parts", "four parts", "one batch row"):
        _case(device, name, LISTS[lists], dtype, layout, ordered=lists != "four parts")


@pytest.mark.gpu
@pytest.mark.parametrize("extent", [70, 32, 16])
@pytest.mark.parametrize("degrees", [[1, 0, 3] * 30, [100, 0, 33, 1, 700]])
def test_output_segments_that_no_path_fills_are_zero(device, jit_on, degrees, extent):
    """w[u] x1[u] x2[] -> out[u] with one of twelve output segments in no path: zero, not what the memory held."""
    from cuequivariance_amd import _lib
    from cuequivariance_amd.cuet.uniform_1d import Uniform1dPlan, run_plan
    from cuequivariance_amd.tables import U1dTables

    E, Z, N = extent, sum(degrees), len(degrees)
    paths = [(k % 3, (k + 1) % 2, k % 4, k if k < 5 else k + 1, 0.5 + k) for k in range(11)]
    tables = U1dTables.make(E, 3, 1, [1, 1, 0, 1], [3, 2, 4, 12], [0, 1, 2, -1], [4], [0, 1, 2, 3], [11], [0], [0],
                            [i for p in paths for i in p[:4]], [p[4] for p in paths])
    plan = Uniform1dPlan(tables, torch.float32, name="unfilled")
    g = torch.Generator().manual_seed(0)
    rows = torch.repeat_interleave(torch.arange(N, dtype=torch.int32), torch.tensor(degrees))
    args = [torch.randn(Z, n, generator=g).to(device) for n in (3 * E, 2 * E, 4)] + [rows.to(device)]
    B, I = _lib.BATCH_DIM_BATCHED, _lib.BATCH_DIM_INDEXED

    def run():
        return run_plan(plan, [B, B, B, I], [-1, -1, -1, 0, N], Z, 1, args)[0]

    want = run().clone()
    assert plan.specialised(device)
    full = [torch.full((N, 12 * E), float("nan"), device=device) for _ in range(4)]  # (the memory of the next output)
    del full
    got = run().reshape(N, 12, E)
    assert (got[:, 5] == 0).all()
    others = [k for k in range(12) if k != 5]
    assert torch.equal(got[:, others], want.reshape(N, 12, E)[:, others])


@pytest.mark.gpu
@pytest.mark.parametrize("name,dtype,layout", [("c32_l2", torch.float32, cue.ir_mul), ("c32_l2", torch.float64, cue.mul_ir), ("c16_l1", torch.float32, cue.mul_ir),
                                               ("c24_l1", torch.float64, cue.ir_mul), ("c5_l1", torch.float32, cue.mul_ir), ("c5_l1", torch.float64, cue.ir_mul)])
def test_a_row_of_the_output_per_batch_row(device, jit_on, name, dtype, layout):
    """Two (four) output rows a wavefront where 32 (16) lanes hold every channel: a last wavefront with some of them, rows read by index."""
    from cuequivariance_amd import cuet
    from oracle.naive import naive_segmented_polynomial, spec_from_polynomial
    from tests.test_mul_ir_addressing import assert_close, to_mul_ir

    ir1, ir2, filt = DESCRIPTORS[name]
    ir1, ir2 = cue.Irreps("O3", ir1), cue.Irreps("O3", ir2)
    m = cuet.ChannelWiseTensorProduct(ir1, ir2, filt, layout=layout, shared_weights=False)
    into1, into3 = [(lambda x, i=i: to_mul_ir(x, i)) if layout == cue.mul_ir else (lambda x: x) for i in (ir1, m.irreps_out)]
    for Z, indexed in ((1, False), (2, True), (3, False), (7, True), (64, False), (1001, False)):
        g = torch.Generator().manual_seed(Z)
        rows = 5 if indexed else Z
        w, x1, x2, cot = (torch.randn(*s, dtype=torch.float64, generator=g).to(dtype).double()
                          for s in ((Z, m.weight_numel), (rows, ir1.dim), (Z, ir2.dim), (Z, m.irreps_out.dim)))
        senders = torch.randint(0, rows, (Z,), generator=g, dtype=torch.int32)
        a = [t.clone().requires_grad_(True) for t in (w, x1, x2)]
        ref = naive_segmented_polynomial(spec_from_polynomial(m.f._polynomial_orig), a, {1: senders} if indexed else {}, {}, {})[0]
        ref_grads = torch.autograd.grad(ref, a, cot)
        b = [t.to(device, dtype).requires_grad_(True) for t in (w, into1(x1), x2)]
        full = [torch.full((Z, m.irreps_out.dim), float("nan"), device=device, dtype=dtype) for _ in range(4)]  # (the memory of the output)
        del full
        out = m(b[1], b[2], b[0], indices_1=senders.to(device) if indexed else None)
        grads = torch.autograd.grad(out, b, into3(cot).to(device, dtype))
        assert m.f.m._plan(dtype).specialised(device)
        for what, got, want in zip(("out", "dw", "dx1", "dx2"), (out, *grads), (into3(ref), ref_grads[0], into1(ref_grads[1]), ref_grads[2])):
            assert_close(got, want, TOL[dtype], what)
