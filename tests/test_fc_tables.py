"""The tables of the fully connected rows kernels (csrc/fc_flex.hip) name parts, weights, rows and packed fragments that exist: every
address a launch would form lies inside its operand, and the packed fragments are each written once."""

import struct

import pytest

from cuequivariance_amd import cue
from cuequivariance_amd.cuet.dense import GeneralFullyConnected, _fc_tables

CASES = [("64x0e+64x1o", "16x0e+16x1o", "64x0e+64x1o"), ("32x0e+16x1o", "4x0e+3x1o", "48x0e+32x1o"), ("32x0e+32x1o", "9x0e+5x1o", "16x0e+80x1o+16x1e"),
         ("80x0e+16x1o+32x2e", "2x0e+1x1o+5x2e", "32x0e+16x1o+48x2e"), ("128x0e+128x1o", "0e+1o", "128x0e+128x1o")]


@pytest.mark.parametrize("x2_mul_ir", [False, True])
@pytest.mark.parametrize("i1,i2,io", CASES)
def test_addresses_lie_inside_the_operands(i1, i2, io, x2_mul_ir):
    irreps = [cue.Irreps("O3", i) for i in (i1, i2, io)]
    e = cue.descriptors.fully_connected_tensor_product(*irreps)
    (fb, fp, xb, xp, dw, coef), tiles, served, most, _, packed = _fc_tables(GeneralFullyConnected(e.polynomial, False, x2_mul_ir), x2_mul_ir)
    numel, w1, n2, wo = (o.size for o in e.polynomial.operations[0][1].operands)

    def rows(blocks, parts, column_tiles, gradient, pieces, steps=5):
        source, result = (wo, w1) if gradient else (w1, wo)
        blocks, parts = list(struct.iter_unpack("<6i", blocks)), list(struct.iter_unpack("<q11iI", parts))
        assert sum(b[5] for b in blocks) == column_tiles and sum(b[4] for b in blocks) == len(parts)
        for c0, n, d, first, count, nt in blocks:
            assert c0 + n * d <= result and nt == -(-n // 32) and first + count <= len(parts)
            for w0, a0, k, ds, co, j0, d2, stride, v, js, vs, wv, mask in parts[first:first + count]:
                assert a0 + k * ds <= source and j0 + (v - 1) * vs + (d2 - 1) * js < n2 and 4 * (co + ds * d * d2) <= len(coef) and mask < 1 << ds * d
                if pieces:
                    last = steps if steps < 5 else k // 16  # (the kernels with the block in registers read all their steps)
                    assert last >= k // 16 and w0 + (v - 1) * wv + ((last - 1) * stride + nt - 1) * 512 + 512 <= pieces * 8
                else:
                    last = (n - 1) * stride + k - 1 if gradient else (k - 1) * stride + n - 1
                    assert w0 + (v - 1) * wv + last < numel

    rows(fb, fp, tiles[0], False, 0)
    rows(xb, xp, tiles[1], True, 0)

    def grads(table, count, group):
        total = 0
        for w0, a0, k, d1, c0, n, d3, co, j0, d2, nt, ntv, stride, v, js, vs, mask in struct.iter_unpack("<q15iI", table):
            assert nt == ntv * -(-k // 64) * -(-v // group) and ntv == -(-n // 64)
            assert a0 + k * d1 <= w1 and c0 + n * d3 <= wo and w0 + (k - 1) * stride + v * n <= numel and j0 + (v - 1) * vs + (d2 - 1) * js < n2
            assert 4 * (co + d1 * d3 * d2) <= len(coef)
            total += nt
        assert total == count

    grads(dw, tiles[2], 1)
    assert (packed is None) == (" " not in i2 and not any(mul > 1 for mul, _ in irreps[1]))
    if packed is not None:
        (pfb, pfp, pxb, pxp, fpk, xpk, pdw), longest, pieces, grad_tiles = packed
        rows(pfb, pfp, tiles[0], False, pieces[0], longest[0])
        rows(pxb, pxp, tiles[1], True, pieces[1], longest[1])
        grads(pdw, grad_tiles, 4)
        for table, total in ((fpk, pieces[0]), (xpk, pieces[1])):
            at = 0
            for src, dst, k, n, sk, sn, v, vs, count, steps in struct.iter_unpack("<2q8i", table):
                assert steps >= k // 16 and dst == at * 8 and count == v * steps * -(-n // 32) * 64 and src + (k - 1) * sk + (n - 1) * sn + (v - 1) * vs < numel
                at += count
            assert at == total
