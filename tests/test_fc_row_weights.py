"""Fully connected tensor product with a weight row per batch row (the product inside the reference's
``FullyConnectedTensorProductConv``, ``cuequivariance_torch/layers/tp_conv_fully_connected.py:216-276``): the kernels of
``cuequivariance_amd/codegen/fullyconnected_rows.py`` against the oracle - forward and the three gradients from the fused
backward, plain batch and gather / scatter by index, both policies for the gathered operand's gradient."""

import pytest
import torch

from cuequivariance_amd import cue, jit
from cuequivariance_amd.codegen import fullyconnected_rows as fcr
from cuequivariance_amd.cue import descriptors
from cuequivariance_amd.tables import U1dTables


def flattened_tables(polynomial):
    from cuequivariance_amd.codegen.registry import flattened_fully_connected_tables

    return flattened_fully_connected_tables(polynomial)


def test_structure_of_the_descriptor():
    i1, i2 = cue.Irreps("O3", "64x0e+64x1o"), cue.Irreps("O3", "0e+1o+2e")
    e = descriptors.fully_connected_tensor_product(i1, i2, i1)
    st = fcr.analyze(e.polynomial)
    assert (st.U, st.Wd, st.width_w, st.width_x1, st.width_x2, st.width_out) == (64, 64, 20480, 256, 9, 256)
    # 0e0e0e, 0e1o1o, 1o0e1o, 1o1o0e, 1o2e1o: non-zeros of the Clebsch-Gordan tensors
    assert [len(b.entries) for b in st.blocks] == [1, 3, 3, 3, 11]
    assert [b.w_off for b in st.blocks] == [4096 * n for n in range(5)]
    t = flattened_tables(e.polynomial)
    assert jit.is_row_weight_fully_connected(t, e.polynomial)
    assert jit._family(t, None, e.polynomial) == "fc_rows" and jit.has_fused_backward(t, None, e.polynomial)
    # not this family: different multiplicities in one operand, a second operand with multiplicity, a channel-wise product
    assert fcr.analyze(descriptors.fully_connected_tensor_product(cue.Irreps("O3", "8x0e+4x1o"), i2, i1).polynomial) is None
    assert fcr.analyze(descriptors.fully_connected_tensor_product(i1, cue.Irreps("O3", "2x0e"), i1).polynomial) is None
    assert fcr.analyze(descriptors.channelwise_tensor_product(i1, i2, "0e+1o").polynomial) is None
    assert fcr.analyze(descriptors.fully_connected_tensor_product(cue.Irreps("O3", "128x0e"), i2, i1).polynomial) is None


def test_unit_compiles_and_registers_under_both_hashes(jit_on):
    i1, i2, i3 = cue.Irreps("O3", "8x0e+8x1o"), cue.Irreps("O3", "0e+1o"), cue.Irreps("O3", "16x0e+16x1o")
    e = descriptors.fully_connected_tensor_product(i1, i2, i3)
    t = flattened_tables(e.polynomial)
    assert not jit._has_spec(t, 0)
    assert jit.ensure_specialised(t, 0, None, origin=e.polynomial)
    assert jit._has_spec(t, 0) and jit._has_spec(t.backward((True, True, True)), 0)


def run_case(device, ir1, ir2, ir3, N, Z, dtype, seed, indexed, sort_receivers=True):
    from cuequivariance_amd import cuet
    from oracle.naive import naive_segmented_polynomial, spec_from_polynomial

    i1, i2, i3 = (cue.Irreps("O3", s) for s in (ir1, ir2, ir3))
    m = cuet.FullyConnectedTensorProduct(i1, i2, i3, layout=cue.ir_mul, shared_weights=False, internal_weights=False,
                                         device=device, dtype=dtype)
    spec = spec_from_polynomial(descriptors.fully_connected_tensor_product(i1, i2, i3).polynomial)
    g = torch.Generator().manual_seed(seed)
    x1 = torch.randn(N if indexed else Z, i1.dim, dtype=torch.float64, generator=g).to(dtype)
    x2 = torch.randn(Z, i2.dim, dtype=torch.float64, generator=g).to(dtype)
    w = torch.randn(Z, m.weight_numel, dtype=torch.float64, generator=g).to(dtype)
    snd = torch.randint(0, max(N, 1), (Z,), generator=g, dtype=torch.int32)
    rcv = torch.randint(0, max(N, 1), (Z,), generator=g, dtype=torch.int32)
    if sort_receivers:
        rcv = torch.sort(rcv)[0]
    cot = torch.randn(N if indexed else Z, i3.dim, dtype=torch.float64, generator=g).to(dtype)
    a = [t.clone().requires_grad_(True) for t in (w, x1, x2)]
    ref = naive_segmented_polynomial(spec, a, {1: snd}, {0: N}, {0: rcv})[0] if indexed else naive_segmented_polynomial(spec, a)[0]
    ref_grads = torch.autograd.grad((ref * cot).sum(), a)
    b = [t.to(device).requires_grad_(True) for t in (w, x1, x2)]
    if indexed:
        out = m(b[1], b[2], b[0], indices_1=snd.to(device), indices_out=rcv.to(device), size_out=N)
    else:
        out = m(b[1], b[2], b[0])
    grads = torch.autograd.grad(out, b, cot.to(device))
    tol = 1e-12 if dtype == torch.float64 else 1e-5

    def close(got, want, what):
        got, want = got.detach().cpu().double(), want.double()
        err = (got - want).abs().max().item()
        assert err <= tol * max(want.abs().max().item(), 1e-30), f"{what}: {err:.3e}"

    close(out, ref, "out")
    for name, p, q in zip(("dw", "dx1", "dx2"), ref_grads, grads):
        close(q, p, name)
    return m


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("deterministic", ["0", "1"])
def test_row_weights_gather_scatter(device, dtype, deterministic, jit_on, monkeypatch):
    """64x0e+64x1o (x) 0e+1o+2e -> 64x0e+64x1o, 60 nodes / 700 edges, x1 gathered by sender, output summed by receiver."""
    monkeypatch.setenv("CUEQ_DETERMINISTIC", deterministic)
    m = run_case(device, "64x0e+64x1o", "0e+1o+2e", "64x0e+64x1o", 60, 700, dtype, seed=21, indexed=True)
    plan = m.f_per_sample.f.m._plan(dtype)
    assert plan.specialised(device) and plan.backward_plan((True, True, True)).specialised(device)
    assert jit._family(plan.tables, plan.polynomial, plan.origin) == "fc_rows"


@pytest.mark.gpu
def test_row_weights_plain_batch_and_unsorted_receivers(device, jit_on):
    run_case(device, "64x0e+64x1o", "0e+1o+2e", "64x0e+64x1o", 0, 300, torch.float32, seed=22, indexed=False)
    run_case(device, "64x0e+64x1o", "0e+1o+2e", "64x0e+64x1o", 500, 64, torch.float64, seed=23, indexed=True, sort_receivers=False)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_row_weights_multiplicities_below_the_wavefront(device, dtype, jit_on):
    """24 input and 40 output channels (lanes beyond them idle), outputs up to l = 2."""
    m = run_case(device, "24x0e+24x1o+24x2e", "0e+1o", "40x0e+40x1o+40x2e", 37, 333, dtype, seed=24, indexed=True)
    assert m.f_per_sample.f.m._plan(dtype).specialised(device)


@pytest.mark.gpu
def test_row_weights_without_batch_rows(device):
    """No edges at all: the output rows are zeros, the gradients have their shapes (the build's unit, no compilation)."""
    from cuequivariance_amd import cuet

    i1, i2 = cue.Irreps("O3", "64x0e+64x1o"), cue.Irreps("O3", "0e+1o+2e")
    m = cuet.FullyConnectedTensorProduct(i1, i2, i1, layout=cue.ir_mul, shared_weights=False, internal_weights=False,
                                         device=device, dtype=torch.float32)
    x1 = torch.randn(5, i1.dim, device=device, requires_grad=True)
    x2 = torch.randn(0, i2.dim, device=device, requires_grad=True)
    w = torch.randn(0, m.weight_numel, device=device, requires_grad=True)
    idx = torch.zeros(0, dtype=torch.int32, device=device)
    out = m(x1, x2, w, indices_1=idx, indices_out=idx, size_out=5)
    assert out.shape == (5, i1.dim) and float(out.detach().abs().sum()) == 0.0
    g1, g2, gw = torch.autograd.grad(out, [x1, x2, w], torch.ones_like(out))
    assert g1.shape == x1.shape and float(g1.abs().sum()) == 0.0 and g2.shape == x2.shape and gw.shape == w.shape
    assert m.f_per_sample.f.m._plan(torch.float32).specialised(device)


MUL_IR_ROWS = [("64x0e+64x1o", "0e+1o+2e", "64x0e+64x1o"), ("24x0e+24x1o+24x2e", "0e+1o", "40x0e+40x1o+40x2e"), ("8x1o", "0e+1o", "16x0e+16x1o")]


@pytest.mark.parametrize("ir1,ir2,ir3", MUL_IR_ROWS[1:])
@pytest.mark.parametrize("in_mul_ir,out_mul_ir", [(True, True), (True, False), (False, True)])
def test_tables_of_mul_ir_rows(ir1, ir2, ir3, in_mul_ir, out_mul_ir):
    """The flattened tables over mul_ir rows are those over ir_mul rows with every scalar of x1 and every segment of the output at the
    place where such a row holds it."""
    from cuequivariance_amd.codegen.registry import flattened_fully_connected_tables

    e = descriptors.fully_connected_tensor_product(*(cue.Irreps("O3", s) for s in (ir1, ir2, ir3)))
    plain, rows = flattened_tables(e.polynomial), fcr.Rows(e.polynomial, in_mul_ir, out_mul_ir)
    t = flattened_fully_connected_tables(rows)
    assert jit._family(t, None, rows) == "fc_rows" and jit._family(t, None, e.polynomial) == (None if out_mul_ir else "fc_rows")

    def place(irreps, mul_ir):  # [(first, distance)] of the components of a row, in ir_mul order
        out, off = [], 0
        for mul, ir in irreps:
            out += [(off + i, ir.dim) if mul_ir else (off + i * mul, 1) for i in range(ir.dim)]
            off += mul * ir.dim
        return out

    U, st = e.inputs[1].irreps[0].mul, fcr.analyze(rows)
    assert st.at_x1 == place(e.inputs[1].irreps, in_mul_ir) and st.at_out == place(e.outputs[0].irreps, out_mul_ir)
    assert t.segment_addressing(3) == st.at_out
    moved = [st.at_x1[c // U][0] + (c % U) * st.at_x1[c // U][1] for c in range(st.width_x1)]
    (_, a), (_, b) = plain.operation(0), t.operation(0)
    assert [((w, moved[x1], x2, out), c) for (w, x1, x2, out), c in a] == [(tuple(i), c) for i, c in b]


@pytest.mark.parametrize("ir1,ir2,ir3", MUL_IR_ROWS)
def test_mul_ir_rows_are_flattened_at_the_cost_of_ir_mul_rows(ir1, ir2, ir3, monkeypatch):
    """What the first call of a module pays for, one object per scalar path and pass over them, is the same in either order of the rows."""
    from cuequivariance_amd.cue import stp

    poly = descriptors.fully_connected_tensor_product(*(cue.Irreps("O3", s) for s in (ir1, ir2, ir3))).polynomial
    made, init = [], stp.Path.__init__

    def counted(self, indices, coefficients):
        made.append(1)
        init(self, indices, coefficients)

    monkeypatch.setattr(stp.Path, "__init__", counted)

    def count(rows):
        made.clear()
        fcr.flatten(rows)
        return len(made)

    assert count(fcr.Rows(poly, True, True)) == count(fcr.Rows(poly))


@pytest.mark.parametrize("compiles", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("which,layouts,served", [
    (0, ("mul_ir", "mul_ir"), (True, True)),    # in the library
    (0, ("mul_ir", "ir_mul"), (False, False)),  # the library has ir_mul rows, one transposition away
    (0, ("ir_mul", "mul_ir"), (False, False)),
    (1, ("mul_ir", "mul_ir"), (False, True)),   # compiled at first use or not at all
    (1, ("mul_ir", "ir_mul"), (False, True)),
])
def test_which_mul_ir_rows_are_taken_as_they_lie(which, layouts, served, dtype, compiles, monkeypatch):
    from cuequivariance_amd import cuet

    i1, i2, i3 = (cue.Irreps("O3", s) for s in (MUL_IR_ROWS[0] if which == 0 else ("20x0e+20x1o", "0e+1o", "12x0e+12x1o")))
    m = cuet.FullyConnectedTensorProduct(i1, i2, i3, layout_in1=cue.IrrepsLayout.as_layout(layouts[0]), layout_in2=cue.mul_ir,
                                         layout_out=cue.IrrepsLayout.as_layout(layouts[1]), shared_weights=False, internal_weights=False)
    monkeypatch.setattr(jit, "_enabled", compiles)
    q, groups = fcr.flatten(m._mul_ir_rows)
    rows = cuet.SegmentedPolynomial(q, method="uniform_1d", options={"origin": m._mul_ir_rows, "segment_groups": groups})
    plan = rows.m._plan(dtype)
    assert m._rows_are_served(plan) == m._rows_are_served(plan) == served[compiles]


@pytest.mark.gpu
@pytest.mark.parametrize("layouts", [("mul_ir", "ir_mul"), ("ir_mul", "mul_ir")])
def test_mixed_row_orders_without_compilation_keep_to_the_library(device, layouts, monkeypatch):
    """One side is transposed and the linked kernels run, forward and backward."""
    from cuequivariance_amd import _lib, cuet

    monkeypatch.setattr(jit, "_enabled", False)
    i1, i2, i3 = (cue.Irreps("O3", s) for s in MUL_IR_ROWS[0])
    more = dict(shared_weights=False, internal_weights=False)
    m = cuet.FullyConnectedTensorProduct(i1, i2, i3, layout_in1=cue.IrrepsLayout.as_layout(layouts[0]), layout_in2=cue.mul_ir,
                                         layout_out=cue.IrrepsLayout.as_layout(layouts[1]), **more)
    same = cuet.FullyConnectedTensorProduct(i1, i2, i3, layout=cue.mul_ir, **more)
    g = torch.Generator(device=device).manual_seed(3)
    x1, x2, w, cot = (torch.randn(77, d, generator=g, device=device) for d in (i1.dim, i2.dim, m.weight_numel, i3.dim))

    def turned(x, irreps, layout, back=False):  # mul_ir rows in the given layout, or back
        if layout == "mul_ir":
            return x
        parts, off = [], 0
        for mul, ir in irreps:
            shape = (-1, ir.dim, mul) if back else (-1, mul, ir.dim)
            parts.append(x[:, off:off + mul * ir.dim].reshape(shape).transpose(1, 2).reshape(-1, mul * ir.dim))
            off += mul * ir.dim
        return torch.cat(parts, 1)

    def step(f, x, c):
        args = [t.clone().requires_grad_() for t in (x, x2, w)]
        out = f(*args)
        return [out.detach(), *torch.autograd.grad(out, args, c)]

    want = step(same, x1, cot)
    _lib.timing_begin()
    got = step(m, turned(x1, i1, layouts[0]).contiguous(), turned(cot, i3, layouts[1]).contiguous())
    names = list(_lib.timing_end())
    assert "segmented_transpose" in names and all(any(n.startswith("fcr_") and f"_{way}_" in n for n in names) for way in ("fwd", "bwd")), names
    plan = m.f_per_sample.f.m._plan(torch.float32)
    assert plan.specialised(device) and plan.backward_plan((True, True, True)).specialised(device)
    got = [turned(got[0], i3, layouts[1], True), turned(got[1], i1, layouts[0], True), got[2], got[3]]
    for a, b in zip(got, want):  # (the same kernels but for the addresses)
        assert (a - b).abs().max().item() <= 1e-6 * b.abs().max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("indexed,deterministic", [(True, "0"), (True, "1"), (False, "0")])
@pytest.mark.parametrize(
    "ir1,ir2,ir3,layouts,dtype",
    [(*MUL_IR_ROWS[0], ("mul_ir", "mul_ir"), torch.float32), (*MUL_IR_ROWS[0], ("mul_ir", "mul_ir"), torch.float64),
     (*MUL_IR_ROWS[1], ("mul_ir", "ir_mul"), torch.float32), (*MUL_IR_ROWS[1], ("ir_mul", "mul_ir"), torch.float32),
     (*MUL_IR_ROWS[2], ("mul_ir", "mul_ir"), torch.float32)],
)
def test_row_weights_on_mul_ir_rows(device, dtype, layouts, ir1, ir2, ir3, indexed, deterministic, jit_on, monkeypatch):
    """Rows in mul_ir as they lie against the oracle on converted rows (float32 1e-5, float64 1e-12 of the largest value, as above), without a
    transposition launch; a hook on the general executor takes the transposing way, with the same result."""
    from cuequivariance_amd import _lib, cuet
    from oracle.naive import naive_segmented_polynomial, spec_from_polynomial

    monkeypatch.setenv("CUEQ_DETERMINISTIC", deterministic)
    i1, i2, i3 = (cue.Irreps("O3", s) for s in (ir1, ir2, ir3))
    m = cuet.FullyConnectedTensorProduct(i1, i2, i3, layout_in1=cue.IrrepsLayout.as_layout(layouts[0]), layout_in2=cue.mul_ir,
                                         layout_out=cue.IrrepsLayout.as_layout(layouts[1]), shared_weights=False, internal_weights=False)
    N, Z = 29, 301

    def turned(x, irreps, layout):  # ir_mul rows in the given layout
        if layout == "ir_mul":
            return x
        parts, off = [], 0
        for mul, ir in irreps:
            parts.append(x[:, off:off + mul * ir.dim].reshape(-1, ir.dim, mul).transpose(1, 2).reshape(-1, mul * ir.dim))
            off += mul * ir.dim
        return torch.cat(parts, 1)

    g = torch.Generator().manual_seed(31)
    x1, x2, w, cot = (torch.randn(*s, dtype=torch.float64, generator=g).to(dtype).double()
                      for s in ((N if indexed else Z, i1.dim), (Z, i2.dim), (Z, m.weight_numel), (N if indexed else Z, i3.dim)))
    snd, rcv = (torch.randint(0, N - 2, (Z,), generator=g, dtype=torch.int32) for _ in range(2))
    a = [t.clone().requires_grad_(True) for t in (w, x1, x2)]
    spec = spec_from_polynomial(descriptors.fully_connected_tensor_product(i1, i2, i3).polynomial)
    ref = naive_segmented_polynomial(spec, a, {1: snd}, {0: N}, {0: rcv})[0] if indexed else naive_segmented_polynomial(spec, a)[0]
    r_w, r_1, r_2 = torch.autograd.grad(ref, a, cot)
    want = [turned(ref.detach(), i3, layouts[1]), r_w, turned(r_1, i1, layouts[0]), r_2]
    b = [t.to(dtype).to(device).requires_grad_(True) for t in (w, turned(x1, i1, layouts[0]), x2)]
    gd = turned(cot, i3, layouts[1]).to(dtype).to(device)
    more = dict(indices_1=snd.to(device), indices_out=rcv.to(device), size_out=N) if indexed else {}

    def step():
        out = m(b[1], b[2], b[0], **more)
        return (out, *torch.autograd.grad(out, b, gd))

    _lib.load().cueq_timing_begin()
    got = step()
    torch.cuda.synchronize()
    names = dict(_lib.timing_end())
    assert "segmented_transpose" not in names, names
    plan = m.per_sample_rows.m._plan(dtype)
    assert plan.specialised(device) and plan.backward_plan((True, True, True)).specialised(device)
    called = []
    m.f_per_sample.register_forward_hook(lambda *_: called.append(1))
    again = step()
    assert called
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    for what, p, q, r in zip(("out", "dw", "dx1", "dx2"), got, again, want):
        assert p.shape == q.shape == r.shape
        for t in (p, q):
            err = (t.detach().cpu().double() - r).abs().max().item()
            assert err <= tol * r.abs().max().item(), (what, err)


@pytest.mark.gpu
def test_mul_ir_rows_without_batch_rows(device):
    """No edges at all on the default layout: the output rows are zeros, the gradients have their shapes (the build's unit)."""
    from cuequivariance_amd import cuet

    i1, i2 = cue.Irreps("O3", "64x0e+64x1o"), cue.Irreps("O3", "0e+1o+2e")
    m = cuet.FullyConnectedTensorProduct(i1, i2, i1, layout=cue.mul_ir, shared_weights=False, internal_weights=False)
    x1 = torch.randn(5, i1.dim, device=device, requires_grad=True)
    x2 = torch.randn(0, i2.dim, device=device, requires_grad=True)
    w = torch.randn(0, m.weight_numel, device=device, requires_grad=True)
    idx = torch.zeros(0, dtype=torch.int32, device=device)
    out = m(x1, x2, w, indices_1=idx, indices_out=idx, size_out=5)
    assert out.shape == (5, i1.dim) and float(out.detach().abs().sum()) == 0.0
    g1, g2, gw = torch.autograd.grad(out, [x1, x2, w], torch.ones_like(out))
    assert g1.shape == x1.shape and float(g1.abs().sum()) == 0.0 and g2.shape == x2.shape and gw.shape == w.shape
    assert m.f_per_sample.f is None  # (the rows were taken as they lie)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("product,compiles,taken", [
    (MUL_IR_ROWS[0], False, True), (MUL_IR_ROWS[0], True, True),
    (("4x1o", "0e+1o", "12x0e+12x1o"), False, False),  # (not in the library: without compilation its rows are transposed)
    (MUL_IR_ROWS[2], True, True),
])
def test_second_derivatives_on_mul_ir_rows(device, product, compiles, taken, dtype, jit_on):
    """Gradients of a function of the output and of its first gradients, against the oracle in float64 (float32: sums over 64 x 64 and
    over 11 products of three random factors, 2e-5 of the largest value)."""
    from cuequivariance_amd import _lib, cuet
    from oracle.naive import naive_segmented_polynomial, spec_from_polynomial

    jit.enable(compiles)  # (the fixture brings the previous state back)
    i1, i2, i3 = (cue.Irreps("O3", s) for s in product)
    m = cuet.FullyConnectedTensorProduct(i1, i2, i3, layout=cue.mul_ir, shared_weights=False, internal_weights=False)
    N, Z = 4, 9
    g = torch.Generator().manual_seed(8)
    r = lambda *s: torch.randn(*s, dtype=torch.float64, generator=g).to(dtype).double()
    x1, x2, w, cot = r(N, i1.dim), r(Z, i2.dim), r(Z, m.weight_numel), r(N, i3.dim)
    snd, rcv = (torch.randint(0, N, (Z,), generator=g, dtype=torch.int32) for _ in range(2))
    inner = [r(*t.shape) for t in (w, x1, x2)]

    def swapped(x, irreps, back):  # mul_ir rows as ir_mul rows, or back
        parts, off = [], 0
        for mul, ir in irreps:
            shape = (-1, ir.dim, mul) if back else (-1, mul, ir.dim)
            parts.append(x[:, off:off + mul * ir.dim].reshape(shape).transpose(1, 2).reshape(-1, mul * ir.dim))
            off += mul * ir.dim
        return torch.cat(parts, 1)

    spec = spec_from_polynomial(descriptors.fully_connected_tensor_product(i1, i2, i3).polynomial)

    def oracle(w, x1, x2):
        return swapped(naive_segmented_polynomial(spec, [w, swapped(x1, i1, False), x2], {1: snd}, {0: N}, {0: rcv})[0], i3, True)

    def ours(w, x1, x2):
        return m(x1, x2, w, indices_1=snd.to(device), indices_out=rcv.to(device), size_out=N)

    def step(f, args, c, inner):
        args = [t.clone().requires_grad_() for t in args]
        first = torch.autograd.grad(f(*args), args, c, create_graph=True)
        return torch.autograd.grad(first, args, inner)

    want = step(oracle, (w, x1, x2), cot, inner)
    to = lambda t: t.to(dtype).to(device)
    _lib.timing_begin()
    got = step(ours, tuple(map(to, (w, x1, x2))), to(cot), list(map(to, inner)))
    assert ("segmented_transpose" in _lib.timing_end()) == (not taken)
    tol = 1e-12 if dtype == torch.float64 else 2e-5
    for a, b in zip(got, want):
        assert (a.cpu().double() - b).abs().max().item() <= tol * b.abs().max().item()
