"""``FullyConnectedTensorProductConv(reduce="mean")`` on the degrees of the product's grouping (``csrc/row_scale.hip``) against PyTorch's
counting: element types, widths that are no multiple of a wavefront, rows that collect nothing, unsorted and 64-bit ids, and
derivatives."""

import pytest
import torch

from cuequivariance_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,width", [(1, 1), (7, 65), (300, 256), (513, 1001)])
def test_mean_is_the_quotient_by_the_degree(device, rows, width, dtype):
    g = torch.Generator().manual_seed(rows)
    ids = torch.randint(0, max(1, rows - 1), (5 * rows,), generator=g, dtype=torch.int64 if rows % 2 else torch.int32).to(device)  # (the last row stays empty)
    x = torch.randn(rows, width, generator=g, dtype=torch.float64).to(device, dtype).requires_grad_(True)
    cot = torch.randn(rows, width, generator=g, dtype=torch.float64).to(device, dtype)
    degree = torch.bincount(ids.long(), minlength=rows).clamp(min=1).double().unsqueeze(1)
    out = _lib.host().rows_mean(x, ids)
    assert torch.equal(out, (x.detach().double() / degree).to(dtype))  # (a quotient rounded once more from 64 bits is the quotient rounded once)
    (grad,) = torch.autograd.grad(out, x, cot, create_graph=True)
    assert torch.equal(grad, (cot.double() / degree).to(dtype))
    y = cot.clone().requires_grad_(True)  # the derivative of the gradient with respect to the cotangent is the mean again
    (grad,) = torch.autograd.grad(_lib.host().rows_mean(x, ids), x, y, create_graph=True)
    (again,) = torch.autograd.grad(grad, y, cot.t().contiguous().t())
    assert torch.equal(again, (cot.double() / degree).to(dtype))


def test_calls_that_are_not_plain_are_left_to_pytorch(device):
    x, ids = torch.randn(4, 3, device=device), torch.tensor([0, 1, 1, 3], device=device)
    mean = _lib.host().rows_mean
    assert mean(x, ids) is not None
    assert mean(x, ids.float()) is None and mean(x.cpu(), ids.cpu()) is None and mean(x[0], ids) is None and mean(x, torch.stack([ids, ids], 1)[:, 0]) is None
    with torch.inference_mode():
        fresh = ids.clone()
    assert mean(x, fresh) is None
