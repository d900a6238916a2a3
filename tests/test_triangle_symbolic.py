"""The triangle update traced with a symbolic side: one program for every length (what the forward keeps for the backward is sized in
symbolic arithmetic), on the CPU with fake tensors and on the GPU against the eager call."""

import pytest
import torch

D = 64


class Update(torch.nn.Module):
    def __init__(self, direction):
        super().__init__()
        self.direction = direction

    def forward(self, x, mask, p_in, g_in, p_out, g_out, norm):
        from cuequivariance_amd import cuet

        return cuet.triangle_multiplicative_update(x, self.direction, mask, norm_in_weight=norm, p_in_weight=p_in, g_in_weight=g_in, p_out_weight=p_out,
                                                   g_out_weight=g_out)


def arguments(n, device, dtype, make=torch.empty):
    return tuple(make(*s, device=device, dtype=dtype) for s in ((1, n, n, D), (1, n, n), (2 * D, D), (2 * D, D), (D, D), (D, D), (D,)))


def exported(args, direction="outgoing"):
    n = torch.export.Dim("n", min=4, max=2048)
    return torch.export.export(Update(direction), args, dynamic_shapes=({1: n, 2: n}, {1: n, 2: n}, None, None, None, None, None))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [96, 67])
def test_export_with_a_dynamic_side(n, dtype):
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode(allow_non_fake_inputs=True):
        program = exported(arguments(n, "cuda", dtype))
    side, = program.range_constraints
    assert program.range_constraints[side].lower == 4 and program.range_constraints[side].upper == 2048


def test_the_kept_bytes_are_enough():
    """The size in closed form against the library's, over forms (mapped, copied, none padded) and types."""
    from cuequivariance_amd import _lib
    from cuequivariance_amd.cuet.triangle import _CODE, _saved_bytes

    lib = _lib.load()
    for dtype, code in _CODE.items():
        for b in (1, 3):
            for n in (1, 2, 7, 8, 63, 64, 65, 130, 391, 512):
                for d in (32, 64, 96, 128, 288):
                    needed = lib.cueq_trimul_saved_bytes(code, b, n, d, d)
                    size = 2 if dtype != torch.float32 else 4
                    assert needed <= _saved_bytes(torch.empty(b, n, n, d, dtype=dtype, device="meta")) <= needed + 2 * b * (n + 8) ** 2 * d * size + 300_000


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_program_for_every_length(device, dtype):
    torch.manual_seed(2)
    normal = lambda *s, device, dtype: torch.randn(*s, device=device, dtype=dtype) * (s[-1] ** -0.5 if len(s) == 2 else 1)
    program, frames = exported(arguments(40, device, dtype, normal), "incoming").module(), []

    def backend(graph, example_inputs):
        frames.append(graph)
        return graph.forward

    eager = Update("incoming")
    compiled = torch.compile(eager, backend=backend, dynamic=True)
    for n in (40, 67, 33, 96):  # (none of them D or 2 D: equal extents are taken for one symbol)
        args = [a.requires_grad_(True) for a in arguments(n, device, dtype, normal)]
        wanted = [args[0], *args[2:]]
        out = eager(*args)
        cot = torch.randn_like(out)
        want = torch.autograd.grad(out, wanted, cot)
        assert torch.equal(program(*args), out)
        got_out = compiled(*args)
        assert torch.equal(got_out, out)
        for a, b in zip(torch.autograd.grad(got_out, wanted, cot), want):
            assert torch.equal(a, b)
    assert len(frames) == 1
