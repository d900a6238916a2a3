"""The work whose speed is followed from version to version: what equivariant networks and pair-representation models have
this package do, through its public modules.

A case is a dict of plain values: the ``kind`` of operation, its sizes, the element type and the ``way`` it is run -
``"forward"`` (inference), ``"train"`` (forward and every gradient a training step asks for) or, for the triangle update,
``"input"`` (forward and the gradient of the pair tensor alone).  ``listed()`` holds one to three cases per kind, ``draw``
gives others over the same ranges, ``prepare`` makes the module and its inputs, ``run`` is one pass.

Kinds
  edge       indexed channel-wise product of a MACE-style interaction: gather by sender, product with the harmonics of the
             edge under per-edge weights, sum onto the receiver (``cuet.ChannelWiseTensorProduct``)
  basis      product basis of MACE (``cuet.SymmetricContraction``)
  linear     equivariant linear layer on node features (``cuet.Linear``)
  fully      fully connected product with attributes of multiplicity one (``cuet.FullyConnectedTensorProduct``)
  general    the same with a second operand of any multiplicity
  conv       message passing with a weight row per edge (``cuet.layers.FullyConnectedTensorProductConv``)
  triangle   triangle multiplicative update of a pair tensor (``cuet.triangle_multiplicative_update``)
  forces     one interaction layer under force training: energies, their gradient with the graph kept, and the gradient of
             a loss on both (a second backward through every module)
"""

from __future__ import annotations

import math

import torch

from cuequivariance_amd import cue, cuet

DEVICE = "cuda"
DTYPES = {"fp32": torch.float32, "fp64": torch.float64, "bf16": torch.bfloat16, "fp16": torch.float16}
ELEMENTS = 10  # chemical elements a product basis keeps weights for


def listed():
    return [
        # one drug-sized molecule: the step of a small simulation or of a small batch, all latency
        dict(name="edge_molecule", kind="edge", mul=32, lmax=2, nodes=31, edges=622, layout="mul_ir", ordered=True, dtype="fp32", way="train"),
        # the interaction block of a medium MACE model on a few thousand atoms (the benchmark of this repository)
        dict(name="edge_100k", kind="edge", mul=128, lmax=3, nodes=5000, edges=100_000, layout="ir_mul", ordered=True, dtype="fp32", way="train"),
        # the same block in mixed precision, in the default layout, on a ragged neighbour list
        dict(name="edge_40k_bf16", kind="edge", mul=128, lmax=3, nodes=2017, edges=40_009, layout="mul_ir", ordered=True, dtype="bf16", way="train"),
        # the product basis behind such a block
        dict(name="basis_20k", kind="basis", mul=128, lmax=3, lout=1, nodes=20_011, layout="mul_ir", dtype="fp32", way="train"),
        # the linear layer of that model while it only predicts
        dict(name="linear_5k_forward", kind="linear", mul=128, lmax=2, rows=5003, layout="mul_ir", dtype="fp32", way="forward"),
        # a linear layer on a large training batch in mixed precision
        dict(name="linear_200k_bf16", kind="linear", mul=128, lmax=2, rows=200_000, layout="ir_mul", dtype="bf16", way="train"),
        # a fully connected product with shared weights (NequIP / skip connections with attributes)
        dict(name="fully_50k", kind="fully", mul=64, lmax=1, l2=2, rows=50_000, layout="mul_ir", dtype="fp32", way="train"),
        # two feature tensors multiplied with each other
        dict(name="general_12k_bf16", kind="general", mul=64, mul2=16, lmax=1, rows=12_501, layout="ir_mul", dtype="bf16", way="train"),
        # a convolution with a weight row per edge (DiffDock-style)
        dict(name="conv_12k", kind="conv", mul=64, lmax=1, l2=2, nodes=1203, edges=12_007, layout="ir_mul", dtype="fp32", way="train"),
        # the pair stack at a crop of 512 residues (the benchmark of this repository)
        dict(name="triangle_512_bf16", kind="triangle", n=512, dim=128, batch=1, outgoing=True, dtype="bf16", way="input"),
        # training on a protein as long as it is: an odd length, every weight with a gradient
        dict(name="triangle_391_bf16", kind="triangle", n=391, dim=128, batch=1, outgoing=False, dtype="bf16", way="train"),
        # energy and force training of one interaction layer on a batch of molecules
        dict(name="forces_9k", kind="forces", mul=64, lmax=1, nodes=451, edges=9001, layout="mul_ir", dtype="fp32", way="train"),
    ]


def _between(rng, low, high):
    """A whole number of [low, high], spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["edge", "edge", "basis", "linear", "fully", "general", "conv", "triangle", "triangle", "forces"])
    layout = rng.choice(["mul_ir", "ir_mul"])
    way = rng.choice(["train", "train", "forward"])
    if kind == "edge":
        mul, lmax = rng.choice([32, 64, 128]), rng.choice([1, 2, 3])
        dtype = rng.choice(["fp32", "fp32", "fp32", "bf16", "fp64"])
        edges = _between(rng, 300, 50_000 if dtype == "fp64" else 100_000)
        return dict(kind=kind, mul=mul, lmax=lmax, nodes=max(8, edges // rng.randint(8, 40)), edges=edges, layout=layout,
                    ordered=rng.random() < 0.75, dtype=dtype, way=way)
    if kind == "basis":
        mul, lmax = rng.choice([(32, 2), (64, 2), (128, 2), (128, 3)])
        return dict(kind=kind, mul=mul, lmax=lmax, lout=rng.choice([0, 1]), nodes=_between(rng, 30, 50_000), layout=layout,
                    dtype=rng.choice(["fp32", "fp32", "bf16"]), way=way)
    if kind == "linear":
        mul, lmax, dtype = rng.choice([32, 64, 128]), rng.choice([1, 2, 3]), rng.choice(["fp32", "bf16", "fp16"])
        width = mul * (lmax + 1) ** 2 * (4 if dtype == "fp32" else 2)
        return dict(kind=kind, mul=mul, lmax=lmax, rows=_between(rng, 30, min(200_000, 450_000_000 // width)), layout=layout, dtype=dtype, way=way)
    if kind == "fully":
        return dict(kind=kind, mul=rng.choice([32, 64, 128]), lmax=1, l2=rng.choice([1, 2]), rows=_between(rng, 100, 50_000), layout=layout,
                    dtype=rng.choice(["fp32", "bf16", "fp16"]), way=way)
    if kind == "general":
        return dict(kind=kind, mul=rng.choice([32, 64]), mul2=rng.choice([4, 8, 16]), lmax=1, rows=_between(rng, 100, 12_500), layout=layout,
                    dtype=rng.choice(["fp32", "bf16"]), way=way)
    if kind == "conv":
        edges = _between(rng, 300, 12_000)
        return dict(kind=kind, mul=rng.choice([32, 48, 64]), lmax=1, l2=rng.choice([1, 2]), nodes=max(8, edges // rng.randint(4, 20)), edges=edges,
                    layout=layout, dtype="fp32", way=way)
    if kind == "triangle":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        n = _between(rng, 48, 384 if dtype == "fp32" else 512)
        return dict(kind=kind, n=n, dim=rng.choice([64, 128]), batch=2 if n < 128 else 1, outgoing=rng.random() < 0.5, dtype=dtype,
                    way=rng.choice(["forward", "input", "train"]))
    edges = _between(rng, 300, 20_000)
    return dict(kind="forces", mul=rng.choice([32, 64]), lmax=1, nodes=max(8, edges // rng.randint(10, 30)), edges=edges, layout=layout,
                dtype="fp32", way="train")


# ---------------------------------------------------------------------------------------------------- modules and inputs
def _irreps(mul, lmax):
    return cue.Irreps("O3", "+".join(f"{mul}x{l}{'eo'[l % 2]}" for l in range(lmax + 1)))


def _names(lmax):
    return [f"{l}{'eo'[l % 2]}" for l in range(lmax + 1)]


def _module(case):
    """The module of a case (of "forces": its four modules) without the seeded weights."""
    kind, layout, dtype = case["kind"], cue.IrrepsLayout.as_layout(case.get("layout", "ir_mul")), DTYPES[case["dtype"]]
    if kind == "edge":
        return cuet.ChannelWiseTensorProduct(_irreps(case["mul"], case["lmax"]), _irreps(1, case["lmax"]), "+".join(_names(case["lmax"])),
                                             layout=layout, shared_weights=False, internal_weights=False, device=DEVICE, dtype=dtype)
    if kind == "basis":
        return cuet.SymmetricContraction(_irreps(case["mul"], case["lmax"]), _irreps(case["mul"], case["lout"]), 3, ELEMENTS, layout=layout,
                                         device=DEVICE, dtype=dtype)
    if kind == "linear":
        irreps = _irreps(case["mul"], case["lmax"])
        return cuet.Linear(irreps, irreps, layout=layout, internal_weights=False, device=DEVICE, dtype=dtype)
    if kind in ("fully", "general"):
        irreps = _irreps(case["mul"], case["lmax"])
        second = _irreps(1, case["l2"]) if kind == "fully" else _irreps(case["mul2"], case["lmax"])
        return cuet.FullyConnectedTensorProduct(irreps, second, irreps, layout=layout, internal_weights=False, device=DEVICE, dtype=dtype)
    if kind == "conv":
        irreps = _irreps(case["mul"], case["lmax"])
        return cuet.layers.FullyConnectedTensorProductConv(irreps, _irreps(1, case["l2"]), irreps, batch_norm=False, layout=layout)
    assert kind == "forces"
    mul, feats = case["mul"], _irreps(case["mul"], case["lmax"])
    tp = cuet.ChannelWiseTensorProduct(feats, _irreps(1, 3), "0e+1o+2e", layout=layout, shared_weights=False, internal_weights=False,
                                       device=DEVICE, dtype=dtype)
    # (rows in mul_ir: neighbouring blocks of one irrep are one block of a larger multiplicity, and models say so)
    hidden, mixed = _irreps(mul, 2), tp.irreps_out.simplify() if layout == cue.mul_ir else tp.irreps_out
    return {"sh": cuet.SphericalHarmonics([0, 1, 2, 3], normalize=True, device=DEVICE), "tp": tp,
            "linear": cuet.Linear(mixed, hidden, layout=layout, internal_weights=False, device=DEVICE, dtype=dtype),
            "basis": cuet.SymmetricContraction(hidden, _irreps(mul, 0), 3, ELEMENTS, layout=layout, device=DEVICE, dtype=dtype)}


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    dtype, train, kind = DTYPES[case["dtype"]], case["way"] == "train", case["kind"]

    def normal(*shape, grad=True, scale=1.0):
        made_in = torch.float64 if dtype == torch.float64 else torch.float32
        x = torch.randn(*shape, device=DEVICE, generator=g, dtype=made_in)
        return (x if scale == 1.0 else x * scale).to(dtype).requires_grad_(grad and train)

    def nodes_of_edges(ordered=True):
        made = torch.randint(0, case["nodes"], (2, case["edges"]), device=DEVICE, generator=g, dtype=torch.int32)
        senders, receivers = made[0].contiguous(), made[1].contiguous()
        return senders, torch.sort(receivers)[0] if ordered else receivers

    def seeded(basis):
        with torch.no_grad():
            basis.weight.copy_(normal(*basis.weight.shape, grad=False, scale=basis.weight.shape[1] ** -0.5))
        return basis

    s = {"kind": kind, "way": case["way"]}
    if kind == "edge":
        m = _module(case)
        senders, receivers = nodes_of_edges(case["ordered"])
        vectors = torch.nn.functional.normalize(torch.randn(case["edges"], 3, device=DEVICE, generator=g), dim=1)
        harmonics = cuet.SphericalHarmonics(list(range(case["lmax"] + 1)), normalize=False, device=DEVICE)
        with torch.no_grad():
            attributes = harmonics(vectors).to(dtype)
        s.update(m=m, args=(normal(case["nodes"], m.irreps_in1.dim), attributes.requires_grad_(train), normal(case["edges"], m.weight_numel)),
                 more=dict(indices_1=senders, indices_out=receivers, size_out=case["nodes"]), cot=normal(case["nodes"], m.irreps_out.dim, grad=False))
    elif kind == "basis":
        m = seeded(_module(case))
        elements = torch.randint(0, ELEMENTS, (case["nodes"],), device=DEVICE, generator=g, dtype=torch.int32)
        s.update(m=m, args=(normal(case["nodes"], m.irreps_in.dim), elements), more={}, cot=normal(case["nodes"], m.irreps_out.dim, grad=False),
                 parameters=(m.weight,))
    elif kind == "linear":
        m = _module(case)
        s.update(m=m, args=(normal(case["rows"], m.irreps_in.dim), normal(1, m.weight_numel)), more={}, cot=normal(case["rows"], m.irreps_out.dim, grad=False))
    elif kind in ("fully", "general"):
        m = _module(case)
        s.update(m=m, args=(normal(case["rows"], m.irreps_in1.dim), normal(case["rows"], m.irreps_in2.dim), normal(1, m.weight_numel)), more={},
                 cot=normal(case["rows"], m.irreps_out.dim, grad=False))
    elif kind == "conv":
        m = _module(case)
        graph = nodes_of_edges()
        s.update(m=m, args=(normal(case["nodes"], m.in_irreps.dim), normal(case["edges"], m.sh_irreps.dim), normal(case["edges"], m.tp.weight_numel)),
                 more=dict(graph=(graph, (case["nodes"], case["nodes"]))), cot=normal(case["nodes"], m.out_irreps.dim, grad=False))
    elif kind == "triangle":
        n, d, b = case["n"], case["dim"], case["batch"]
        x = normal(b, n, n, d, grad=False).requires_grad_(case["way"] != "forward")
        weights = dict(norm_in_weight=(1 + normal(d, grad=False, scale=0.1)).requires_grad_(train), norm_in_bias=normal(d, scale=0.1),
                       p_in_weight=normal(2 * d, d, scale=d ** -0.5), g_in_weight=normal(2 * d, d, scale=d ** -0.5),
                       norm_out_weight=(1 + normal(d, grad=False, scale=0.1)).requires_grad_(train), norm_out_bias=normal(d, scale=0.1),
                       p_out_weight=normal(d, d, scale=d ** -0.5), g_out_weight=normal(d, d, scale=d ** -0.5))
        mask = (torch.rand(b, n, n, device=DEVICE, generator=g) < 0.9).to(dtype)
        s.update(m=cuet.triangle_multiplicative_update, args=(x,), parameters=tuple(weights.values()),
                 more=dict(weights, direction="outgoing" if case["outgoing"] else "incoming", mask=mask), cot=normal(b, n, n, d, grad=False))
    else:
        m = _module(case)
        seeded(m["basis"])
        senders, receivers = nodes_of_edges()
        nodes, edges = case["nodes"], case["edges"]
        s.update(m=m, vectors=normal(edges, 3), features=normal(nodes, m["tp"].irreps_in1.dim), radial=normal(edges, m["tp"].weight_numel),
                 mixing=normal(1, m["linear"].weight_numel), elements=torch.randint(0, ELEMENTS, (nodes,), device=DEVICE, generator=g, dtype=torch.int32),
                 senders=senders, receivers=receivers, nodes=nodes, ones=torch.ones(nodes, m["basis"].irreps_out.dim, device=DEVICE, dtype=dtype),
                 cots=(normal(nodes, m["basis"].irreps_out.dim, grad=False), normal(edges, 3, grad=False),
                       normal(edges, m["tp"].weight_numel, grad=False)))
    return s


def _forces(s):
    """Energies, their gradient towards the edge vectors and the radial weights (where the forces come from), and the
    gradient of a loss on all of them (its cotangents given) for the features, the radial weights and the module weights."""
    m = s["m"]
    y = m["sh"](s["vectors"])
    a = m["tp"](s["features"], y, s["radial"], indices_1=s["senders"], indices_out=s["receivers"], size_out=s["nodes"])
    energies = m["basis"](m["linear"](a, s["mixing"]), s["elements"])
    slopes = torch.autograd.grad(energies, [s["vectors"], s["radial"]], s["ones"], create_graph=True)
    wanted = [s["features"], s["radial"], s["mixing"], m["basis"].weight]
    return [energies, *slopes, *torch.autograd.grad([energies, *slopes], wanted, list(s["cots"]))]


def run(s):
    if s["kind"] == "forces":
        return _forces(s)
    if s["way"] == "forward":
        with torch.no_grad():
            return [s["m"](*s["args"], **s["more"])]
    out = s["m"](*s["args"], **s["more"])
    wanted = [t for t in (*s["args"], *s.get("parameters", ())) if t.requires_grad]
    return [out, *torch.autograd.grad(out, wanted, s["cot"])]


# ---------------------------------------------------------------------------------------------------- floors and tolerances
def _paths(e):
    """Scalar paths of a product descriptor after its coefficients are flattened."""
    return sum(stp.num_paths for _, stp in e.flatten_coefficient_modes().polynomial.operations)


def _channelwise(mul, l1, l2, lout):
    e = cue.descriptors.channelwise_tensor_product(_irreps(mul, l1), _irreps(1, l2), _irreps(1, lout))
    return e.inputs[0].dim, e.inputs[1].dim, e.inputs[2].dim, e.outputs[0].dim, _paths(e)


def _fully_connected(first, second, out):
    e = cue.descriptors.fully_connected_tensor_product(first, second, out)
    stp = e.polynomial.operations[0][1]
    # a path is a (u v) x w block of weights; each component of its output irrep is one such contraction per row
    products = sum(math.prod(stp.get_segment_shape(0, path)) * out[path.indices[3]].ir.dim for path in stp.paths)
    return e.inputs[0].dim, products


def _basis(mul, lin, lout):
    e, _ = cue.mace.symmetric_contraction(_irreps(mul, lin), _irreps(mul, lout), range(1, 4))
    # a scalar path of degree n multiplies n + 1 factors and adds: n + 1 operations or so for every channel
    return e.inputs[0].dim, sum(stp.num_paths * stp.num_operands for _, stp in e.flatten_coefficient_modes().polynomial.operations)


def work(case):
    """Bytes: every input read and every output written once per pass (forward; backward).  Flops: two per multiply-add of
    the contraction, once for the forward and once for every gradient."""
    kind, train, size = case["kind"], case["way"] == "train", torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    if kind == "edge":
        w, d1, d2, d3, paths = _channelwise(case["mul"], case["lmax"], case["lmax"], case["lmax"])
        n, e = case["nodes"], case["edges"]
        forward = (e * (w + d2) + n * (d1 + d3)) * size + 8 * e
        backward = (2 * e * (w + d2) + n * (2 * d1 + d3)) * size + 8 * e
        flops = 2 * e * case["mul"] * paths
        return {"bytes": forward + (backward if train else 0), "flops": flops * (4 if train else 1)}
    if kind == "basis":
        w, ops = _basis(case["mul"], case["lmax"], case["lout"])
        n, din, dout = case["nodes"], case["mul"] * (case["lmax"] + 1) ** 2, case["mul"] * (case["lout"] + 1) ** 2
        forward, backward = (n * (din + dout) + ELEMENTS * w) * size + 4 * n, (n * (2 * din + dout) + 2 * ELEMENTS * w) * size + 4 * n
        return {"bytes": forward + (backward if train else 0), "flops": n * case["mul"] * ops * (3 if train else 1)}
    if kind == "linear":
        comps, mul, rows = (case["lmax"] + 1) ** 2, case["mul"], case["rows"]
        w, width = mul * mul * (case["lmax"] + 1), mul * comps
        forward, backward = (2 * rows * width + w) * size, (3 * rows * width + 2 * w) * size
        return {"bytes": forward + (backward if train else 0), "flops": 2 * rows * comps * mul * mul * (3 if train else 1)}
    if kind in ("fully", "general", "conv"):
        irreps = _irreps(case["mul"], case["lmax"])
        second = _irreps(case["mul2"], case["lmax"]) if kind == "general" else _irreps(1, case["l2"])
        w, products = _fully_connected(irreps, second, irreps)
        rows = case["edges"] if kind == "conv" else case["rows"]
        first, weights = (case["nodes"], rows * w) if kind == "conv" else (rows, w)
        forward = first * 2 * irreps.dim + rows * second.dim + weights
        backward = first * 3 * irreps.dim + rows * 2 * second.dim + 2 * weights
        index = 8 * rows if kind == "conv" else 0
        return {"bytes": (forward + (backward if train else 0)) * size + index * (2 if train else 1), "flops": 2 * rows * products * (4 if train else 1)}
    if kind == "triangle":
        n, d, b = case["n"], case["dim"], case["batch"]
        m, w = b * n * n, 6 * d * d + 4 * d
        projections, contraction = 2 * m * d * 6 * d, 2 * b * d * n ** 3
        values, flops = 2 * m * d + m + w, projections + contraction  # the pair tensor, the mask, the weights; the update
        if case["way"] != "forward":  # both factors of the contraction, the input of the projections - and their weights
            values += 3 * m * d + m + w + (w if train else 0)
            flops += (2 if train else 1) * projections + 2 * contraction
        return {"bytes": values * size, "flops": flops}
    assert kind == "forces"
    mul, n, e = case["mul"], case["nodes"], case["edges"]
    w, d1, d2, d3, paths = _channelwise(mul, case["lmax"], 3, 2)
    wb, ops = _basis(mul, 2, 0)
    hidden = 9 * mul
    # inputs and cotangents once, outputs once: the layer as one operation
    values = e * (3 + w) * 2 + n * (d1 + 2 * mul) + e * (3 + w) * 2 + n * d1 + ELEMENTS * wb * 2
    linear = d3 * mul  # one mul x mul block per component of the mixed irreps
    # forward, first gradient and second gradient: 1, 2 and 4 times the contraction
    return {"bytes": values * size + 8 * e + 4 * n, "flops": 2 * 7 * (e * mul * paths + n * linear) + 7 * n * mul * ops + n * hidden}


def tolerance(case):
    if case["dtype"] == "fp64":
        return {"rel": 1e-12}
    if case["dtype"] == "fp32":
        return {"rel": 2e-5 if case["kind"] == "forces" else 1e-5}
    if case["dtype"] == "fp16":
        return {"rel": 3e-3}
    return {"rel": 1.5e-2 if case["kind"] == "triangle" else 1e-2}
