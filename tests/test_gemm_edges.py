"""Products whose last tiles of 128 x 128 are partly filled (``cueq_gemm``): a single tile, one column of tiles, few and many partial tiles
among whole ones, in all four forms of the operands."""

import pytest
import torch

from cuequivariance_amd import _lib

pytestmark = pytest.mark.gpu
CODE = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16}
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-2}  # sums of at most 72 products of unit size; one rounding of the result


@pytest.mark.parametrize("dtype", list(CODE))
@pytest.mark.parametrize("trans_a", [0, 1])
@pytest.mark.parametrize("trans_b", [0, 1])
@pytest.mark.parametrize("M,N,K,batch", [(8, 8, 8, 1), (32, 64, 40, 5), (128, 8, 40, 2), (96, 128, 72, 3), (1160, 128, 40, 1), (136, 264, 72, 2),
                                         (520, 520, 40, 2), (1032, 1032, 40, 1)])
def test_products(device, M, N, K, batch, trans_a, trans_b, dtype):
    g = torch.Generator(device=device).manual_seed(M + N)
    A = torch.randn(batch, *((K, M) if trans_a else (M, K)), device=device, generator=g).to(dtype)
    B = torch.randn(batch, *((K, N) if trans_b else (N, K)), device=device, generator=g).to(dtype)
    C = torch.full((batch, M + 1, N), 7.0, device=device, dtype=dtype)  # (a row between products that nothing may touch)
    _lib.check(_lib.load().cueq_gemm(CODE[dtype], CODE[dtype], trans_a, trans_b, M, N, K, A.data_ptr(), A.shape[2], A[0].numel(), B.data_ptr(), B.shape[2],
                                     B[0].numel(), C.data_ptr(), N, C[0].numel(), batch, 0.5, 0, torch.cuda.current_stream().cuda_stream), "cueq_gemm")
    a, b = A.double().cpu(), B.double().cpu()
    want = 0.5 * (a.transpose(1, 2) if trans_a else a).contiguous() @ (b if trans_b else b.transpose(1, 2)).contiguous()
    assert (C[:, :M].double().cpu() - want).abs().max().item() <= TOL[dtype] * want.abs().max().item()
    assert (C[:, M] == 7).all()
