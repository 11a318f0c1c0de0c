"""GPU parity of the wide matrix-core tile (csrc/tile.hip) against the oracle:
every format at the edges of each tile shape (32 x 32, 64 x 64, 128 x 64 and
128 x 128 rows x tokens), with K split evenly and with a remainder."""
import numpy as np
import pytest

import oracle
from pulsar_amd import formats as fm
from pulsar_amd import kernels as K
from pulsar_amd import synth
from pulsar_amd.formats import (QUANT_IQ2_XXS, QUANT_IQ4_XS, QUANT_Q2_K, QUANT_Q3_K, QUANT_Q4_K, QUANT_Q5_K,
                                QUANT_Q6_K, row_bytes)
from tests.gpu_util import assert_rows_close, down, up, zeros_f32

pytestmark = pytest.mark.gpu
FORMATS = [QUANT_Q4_K, QUANT_Q5_K, QUANT_Q6_K, QUANT_Q2_K, QUANT_Q3_K, QUANT_IQ4_XS, QUANT_IQ2_XXS]


def edge_rows(rows):
    """The first and last rows and those around the tile and wave edges."""
    at = [r + d for r in (0, 16, 32, 64, 128, rows // 2, rows) for d in range(-2, 3)]
    return sorted({r for r in at if 0 <= r < rows})


def xq_rows(n_tok, n, rng, unit):
    """q8_K rows; unit: d = 1 and codes up to +-127, so every dot with unit
    weight scales is an exact integer."""
    if not unit:
        return oracle.quantize_q8_k(rng.standard_normal((n_tok, n)).astype(np.float32))
    nb = n // 256
    qs = rng.integers(-127, 128, (n_tok, nb, 256)).astype(np.int8)
    blk = np.zeros((n_tok, nb, 292), np.uint8)
    blk[..., 0:4] = np.array([1.0], np.float32).view(np.uint8)
    blk[..., 4:260] = qs.view(np.uint8)
    sums = qs.reshape(n_tok, nb, 16, 16).astype(np.int16).sum(-1).astype(np.int16)
    blk[..., 260:292] = sums.view(np.uint8).reshape(n_tok, nb, 32)
    return blk.reshape(n_tok, nb * 292)


def unit_scales(quant, w):
    blk = w.reshape(-1, fm.BLOCK_LAYOUT[quant][1])
    for off in {QUANT_Q4_K: (0, 2), QUANT_Q5_K: (0, 2), QUANT_Q2_K: (80, 82), QUANT_Q6_K: (208,), QUANT_Q3_K: (108,),
                QUANT_IQ4_XS: (0,), QUANT_IQ2_XXS: (0,)}[quant]:
        blk[:, off], blk[:, off + 1] = 0x00, 0x48 if quant == QUANT_IQ2_XXS else 0x3C  # 8 (0.125 d = 1), else 1
    if quant == QUANT_Q6_K:  # the whole range of the int8 scales
        blk[:, 192:208] = synth.rng_for(5, "sc").integers(0, 256, (blk.shape[0], 16), dtype=np.uint8)


def rows_want(quant, w, rb, xq, n, n_tok):
    """(values, bound) of the rows. The tile forms a super-block's value from
    exact integers as yd (fma(-xmin, msum, fl(xd isum))): at most 3 roundings of
    each product's size on its side and 3 on the oracle's, so where the two
    products of a format with mins cancel, |delta| <= 6 2^-24 (P + M) with P the
    sum of |xd yd isum| (the oracle with the mins taken out) and M <= P +
    sum |f_b| that of the min products; 1e-5 sum |f_b| as everywhere covers the
    sums over the super-blocks."""
    want, scale = oracle.rows_dot(w, rb, w.shape[0], xq, n, n_tok, quant, 8)
    bound = scale
    if quant in (QUANT_Q4_K, QUANT_Q5_K, QUANT_Q2_K):
        w0 = w.copy()
        off = 82 if quant == QUANT_Q2_K else 2
        w0.reshape(-1, fm.BLOCK_LAYOUT[quant][1])[:, off:off + 2] = 0
        _, p = oracle.rows_dot(w0, rb, w.shape[0], xq, n, n_tok, quant, 8)
        bound = scale + 6 * 2.0**-24 / 1e-5 * (2 * p + scale)
    return want, scale, bound


# rows x tokens that take each tile shape, ragged in both
SHAPES = [(33, 1500, 512), (1000, 41, 256), (4129, 130, 768), (4130, 500, 256), (4143, 1010, 768), (8200, 19, 1280)]


@pytest.mark.parametrize("quant", FORMATS)
@pytest.mark.parametrize("rows,n_tok,n", SHAPES)
def test_tile_gemm(dev, quant, rows, n_tok, n):
    rng = np.random.default_rng(rows * 31 + n_tok)
    rb = row_bytes(quant, n)
    at = edge_rows(rows)
    for unit in (True, False):
        w = synth.quant_matrix(quant, rows, n, synth.rng_for(rows + n_tok, "tile"))
        if unit:
            unit_scales(quant, w)
        xq = xq_rows(n_tok, n, rng, unit)
        out = zeros_f32((n_tok, rows))
        K.matmul_kq(out, up(w), up(xq), n, rows, n_tok, rb, quant)
        got = down(out)
        want, scale, bound = rows_want(quant, np.ascontiguousarray(w[at]), rb, xq, n, n_tok)
        if unit and n == 256:
            # one super-block: an exact integer where it fits 24 bits (with a
            # min term the two products are integers of their own)
            small = scale < 2**24
            assert small.any() and np.array_equal(got[:, at][small], want[small])
        assert_rows_close(got[:, at], want, bound, f"tile {fm.NAMES[quant]} {rows}x{n} t{n_tok}")
        assert np.isfinite(got).all()
        if n_tok >= 8:
            # every other element: the one-token kernel on the same rows (its
            # sums differ from the tile's by their order alone)
            one = zeros_f32((1, rows))
            for t in (0, n_tok // 2, n_tok - 1):
                K.matmul_kq(one, up(w), up(xq[t]), n, rows, 1, rb, quant)
                ref = down(one)[0]
                assert np.abs(got[t] - ref).max() <= 4e-6 * max(1.0, np.abs(ref).max()) * np.sqrt(n / 256) + 1e-30
