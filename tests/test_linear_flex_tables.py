"""``cueq_linear_flex`` called with tables of its own: what its header takes beyond what the modules ask for."""

import struct

import pytest
import torch

from cuequivariance_amd import _lib

pytestmark = pytest.mark.gpu

CODE = {torch.float32: 0, torch.float16: 2, torch.bfloat16: 3}
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}  # sums of 32 products of unit size; one rounding of the result


def _up(n, to=8):
    return -(-n // to) * to


def _check(device, dtype, blocks, K, rows, mul_ir, transposed=False):
    """``blocks``: (N, D) of the result's blocks, each from a block of K channels of its own; everything between and behind the blocks'
    columns keeps its bits."""
    assert CODE[dtype] == getattr(_lib, {torch.float32: "F32", torch.float16: "F16", torch.bfloat16: "BF16"}[dtype])
    a0 = c0 = w0 = tiles = 0
    packed_blocks, packed_parts, places = b"", b"", []
    for i, (N, D) in enumerate(blocks):
        packed_blocks += struct.pack("<q6i", c0, N, D, i, 1, -(-N // 32), 0)
        packed_parts += struct.pack("<qqif", a0, w0, K, 0.5)
        places.append((a0, c0, w0, N, D))
        a0, c0, w0, tiles = a0 + K * D, _up(c0 + N * D), _up(w0 + K * N), tiles + -(-N // 32)
    lda, ldc = a0, c0 + 8
    g = torch.Generator(device=device).manual_seed(rows + lda)
    A, W = torch.randn(rows, lda, device=device, generator=g).to(dtype), torch.randn(w0, device=device, generator=g).to(dtype)
    C = torch.full((rows, ldc), 7.0, device=device, dtype=dtype)
    on = lambda b: torch.frombuffer(bytearray(b), dtype=torch.uint8).to(device)
    tb, tp = on(packed_blocks), on(packed_parts)
    _lib.check(_lib.load().cueq_linear_flex(CODE[dtype], int(transposed), rows, A.data_ptr(), lda, W.data_ptr(), C.data_ptr(), ldc, tb.data_ptr(), len(blocks),
                                            tp.data_ptr(), tiles, mul_ir, torch.cuda.current_stream().cuda_stream), "cueq_linear_flex")
    kept = torch.ones(ldc, dtype=torch.bool, device=device)
    for a0, c0, w0, N, D in places:
        w = W[w0: w0 + K * N].double()
        w = w.reshape(N, K).T if transposed else w.reshape(K, N)
        x = A[:, a0: a0 + K * D].double().reshape(rows, K, D)
        got, want = C[:, c0: c0 + N * D].double().reshape(rows, N, D), torch.stack([0.5 * (x[..., d] @ w) for d in range(D)], 2)
        assert (got - want).abs().max().item() <= TOL[dtype] * want.abs().max().item()
        kept[c0: c0 + N * D] = False
    assert (C[:, kept] == 7).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("mul_ir", [0, 1, 4, 1 + 4])
def test_many_rows_of_blocks_of_several_components(device, mul_ir, transposed, dtype):
    """The row counts from which on blocks of one component take four row tiles a wavefront: whoever names the rows ``ir_mul`` (0) may
    have blocks of more all the same."""
    _check(device, dtype, [(32, 1), (64, 3), (32, 5), (160, 1), (16, 7)], 32, 40_003, mul_ir, transposed)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("said", [2, 2 + 4])
@pytest.mark.parametrize("rows,extents", [(40_003, (32, 64, 16, 160)), (40_003, (96, 224)), (9_001, (96, 16, 224)), (9_001, (32, 64)), (1_501, [32] * 70)])
def test_many_rows_of_blocks_of_one_component(device, rows, extents, said, transposed, dtype):
    """Tiles through LDS four rows high, tiles a wavefront has to itself, one and two rows high, and more blocks than lanes."""
    _check(device, dtype, [(n, 1) for n in extents], 48, rows, said, transposed)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mul_ir,blocks", [(1, [(4, 1), (20, 3), (36, 5), (68, 1), (12, 7)]), (2, [(4, 1), (36, 1), (132, 1)]), (0, [(100, 3), (228, 1)])])
@pytest.mark.parametrize("rows", [700, 12_001, 40_003])
def test_blocks_that_end_in_half_a_piece(device, rows, mul_ir, blocks, dtype):
    """N of 4 in 2-byte elements: a block's last 8 bytes of a row are half of a 16-byte piece, and what lies behind them belongs to nobody."""
    _check(device, dtype, blocks, 32, rows, mul_ir)


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("rows", [2_049, 40_003])
@pytest.mark.parametrize("blocks", [[(96, 3), (96, 1)], [(224, 1), (96, 5)], [(32, 7), (32, 5), (16, 3), (32, 1)]])
def test_three_column_tiles_left_and_one(device, blocks, rows, transposed):
    """Three column tiles beside a multiple of four (a workgroup's fourth wavefront has the last row tile), and blocks of one in 2-byte elements."""
    for dtype in (torch.float32, torch.bfloat16):
        _check(device, dtype, blocks, 48, rows, 1 + 4, transposed)
