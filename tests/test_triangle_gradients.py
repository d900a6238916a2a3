"""The gradients of the triangle update's weights are tensors of their own (storage, version counter), through the modules' way and
through both C entries."""

import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu
NAMES = ["norm_in_weight", "norm_in_bias", "p_in_weight", "p_in_bias", "g_in_weight", "g_in_bias", "norm_out_weight", "norm_out_bias", "p_out_weight",
         "p_out_bias", "g_out_weight", "g_out_bias"]


def arguments(device, dtype, n=37, d=64, do=32):
    g = torch.Generator().manual_seed(n)
    shapes = [(d,), (d,), (2 * d, d), (2 * d,), (2 * d, d), (2 * d,), (d,), (d,), (do, d), (do,), (do, d), (do,)]
    make = lambda *s: (torch.randn(*s, generator=g) * (d ** -0.5 if len(s) == 2 else 1)).to(dtype).to(device)
    return make(1, n, n, d), [make(*s) for s in shapes], make(1, n, n, do)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("wanted", [range(12), (2, 8, 11), (0,)])
def test_gradients_of_their_own(device, dtype, wanted):
    from cuequivariance_amd import cuet

    x, weights, dout = arguments(device, dtype)
    inputs = [weights[i].requires_grad_(True) for i in wanted]
    out = cuet.triangle_multiplicative_update(x, "outgoing", **dict(zip(NAMES, weights)))
    grads = torch.autograd.grad(out, inputs, dout)
    for g, w in zip(grads, inputs):
        assert g.shape == w.shape and g.is_contiguous() and g.data_ptr() % 16 == 0
        assert g.untyped_storage().nbytes() == g.numel() * g.element_size() and g._base is None
    kept = [g.clone() for g in grads]
    versions = [g._version for g in grads]
    grads[0].add_(1)
    assert [g._version for g in grads[1:]] == versions[1:]
    assert all(torch.equal(a, b) for a, b in zip(grads[1:], kept[1:]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("need", [0xFFF, 0x104, 0x800])
def test_both_entries(device, dtype, need):
    """One buffer, and a tensor per gradient (the others are not touched)."""
    from cuequivariance_amd import _lib
    from cuequivariance_amd.cuet.triangle import _CODE

    lib, code = _lib.load(), _CODE[dtype]
    x, weights, dout = arguments(device, dtype)
    (_, n, _, d), do = x.shape, dout.shape[3]
    stream = torch.cuda.current_stream().cuda_stream
    pointers = (C.c_void_p * 12)(*[w.data_ptr() for w in weights])
    raw = lambda nbytes: torch.empty(max(int(nbytes), 16), dtype=torch.uint8, device=device)
    saved, out = raw(lib.cueq_trimul_saved_bytes(code, 1, n, d, do)), torch.empty_like(dout)
    ws = [raw(lib.cueq_trimul_workspace_bytes(code, 1, n, d, do, back, 1)) for back in (0, 1)]
    _lib.check(lib.cueq_trimul_fwd(code, 1, n, d, do, 1, 1e-5, x.data_ptr(), None, pointers, out.data_ptr(), saved.data_ptr(), ws[0].data_ptr(), ws[0].numel(),
                                   stream), "forward")
    both = []
    for entry in ("buffer", "parts"):
        dx = torch.empty_like(x)
        call = lambda f, grads: _lib.check(f(code, 1, n, d, do, 1, x.data_ptr(), None, pointers, saved.data_ptr(), dout.data_ptr(), dx.data_ptr(), need, grads,
                                             ws[1].data_ptr(), ws[1].numel(), stream), "backward")
        if entry == "buffer":
            buffer = torch.full((lib.cueq_trimul_grads_values(d, do),), 7.0, dtype=dtype, device=device)
            call(lib.cueq_trimul_bwd, buffer.data_ptr())
            order, at, grads = (0, 1, 6, 7, 4, 2, 10, 8, 5, 3, 11, 9), 0, {}
            for i in order:
                grads[i] = buffer[at:at + weights[i].numel()].view(weights[i].shape)
                at += weights[i].numel()
        else:
            grads = {i: torch.full_like(w, 7.0) for i, w in enumerate(weights)}
            call(lib.cueq_trimul_bwd_parts, (C.c_void_p * 12)(*[grads[i].data_ptr() for i in range(12)]))
            assert all(bool((grads[i] == 7).all()) for i in range(12) if not need >> i & 1)
        both.append([dx, *[grads[i] for i in range(12) if need >> i & 1]])
    assert all(torch.equal(a, b) for a, b in zip(*both))
    assert lib.cueq_trimul_bwd_parts(code, 1, n, d, do, 1, x.data_ptr(), None, pointers, saved.data_ptr(), dout.data_ptr(), dx.data_ptr(), 1, (C.c_void_p * 12)(),
                                     ws[1].data_ptr(), ws[1].numel(), stream) != 0  # (a gradient asked for without a place)
