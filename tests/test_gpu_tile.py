"""GPU parity of the wide matrix-core tile (csrc/tile.hip, tile_moe.hip) against
the oracle: every format at the edges of each tile shape (32 x 32, 64 x 64, 128
x 64 and 128 x 128 rows x tokens), with K split evenly and with a remainder, and
the grouped stages over groups of 1 to 150 pairs from both group sources."""
import numpy as np
import pytest
import torch

import oracle
from pulsar_amd import formats as fm
from pulsar_amd import kernels as K
from pulsar_amd import synth
from pulsar_amd.formats import (QUANT_IQ2_XXS, QUANT_IQ4_XS, QUANT_Q2_K, QUANT_Q3_K, QUANT_Q4_K, QUANT_Q5_K,
                                QUANT_Q6_K, row_bytes)
from tests.gpu_util import assert_rows_close, up, zeros_f32
from tests.gpu_util import down as down_np

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
        got = down_np(out)
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
                ref = down_np(one)[0]
                assert np.abs(got[t] - ref).max() <= 4e-6 * max(1.0, np.abs(ref).max()) * np.sqrt(n / 256) + 1e-30


def grouped_case(quant, hidden, ffn, sizes, n_used, rng, down):
    """Experts' matrices, the (token, slot) ids of groups of the given sizes and
    q8_K rows; ids -1 where nothing is routed."""
    E, T = len(sizes), -(-sum(sizes) // n_used) + 3
    rows, cols = (hidden, ffn) if down else (ffn, hidden)
    mats = [synth.quant_matrix(quant, E * rows, cols, synth.rng_for(E * cols + k, "grp")).reshape(E, rows, -1)
            for k in range(1 if down else 2)]
    flat = np.concatenate([np.full(n, e) for e, n in enumerate(sizes)] + [np.full(T * n_used - sum(sizes), -1)])
    ids = rng.permutation(flat).reshape(T, n_used).astype(np.int32)
    x = rng.standard_normal((T * n_used if down else T, cols)).astype(np.float32) * (1.0 if down else 1e-2)
    return mats, ids, oracle.quantize_q8_k(x)


def check_grouped(quant, mats, ids, xq, wts, got, down, cols, what):
    """got [T * n_used][rows] against the oracle, group by group."""
    rb, n_used = row_bytes(quant, cols), ids.shape[1]
    for e in range(mats[0].shape[0]):
        at = np.flatnonzero(ids.reshape(-1) == e)
        if at.size == 0:
            continue
        rows = xq[at] if down else xq[at // n_used]
        vals = [rows_want(quant, m[e], rb, rows, cols, at.size) for m in mats]
        if down:
            assert_rows_close(got[at], vals[0][0], vals[0][2], f"{what} expert {e}")
            continue
        (g, _, bg), (u, _, bu) = vals
        g, u, bg, bu = (v.astype(np.float64) for v in (g, u, 1e-5 * bg, 1e-5 * bu))
        silu, w = g / (1 + np.exp(-g)), np.abs(wts.reshape(-1)[at].astype(np.float64))[:, None]
        # |silu'| <= 1.1; the device's exp, division and two products: 1e-6
        bound = w * (1.1 * bg * (np.abs(u) + bu) + np.abs(silu) * bu) + 1e-6 * np.abs(silu * u) * w + 1e-30
        err = np.abs(got[at] - silu * u * wts.reshape(-1)[at].astype(np.float64)[:, None])
        assert (err <= bound).all(), (what, e, float((err / bound).max()))


# groups of one to three tiles, their edges, and an expert nobody selects
SIZES = [1, 16, 17, 150, 0, 64, 65, 32, 33, 129, 128]


@pytest.mark.parametrize("down", [False, True])
@pytest.mark.parametrize("quant", FORMATS)
def test_tile_grouped(dev, quant, down):
    rng = np.random.default_rng(quant * 2 + down)
    hidden, ffn, n_used = (330, 768, 3) if down else (768, 150, 3)
    mats, ids, xq = grouped_case(quant, hidden, ffn, SIZES, n_used, rng, down)
    T, E = ids.shape[0], len(SIZES)
    rows, cols = (hidden, ffn) if down else (ffn, hidden)
    rb = row_bytes(quant, cols)
    wts = rng.uniform(0.1, 1.0, (T, n_used)).astype(np.float32)
    d_mats, d_xq, d_w = [up(m) for m in mats], up(xq), torch.from_numpy(wts).to(dev)
    ptr = [m.data_ptr() for m in d_mats]
    # a caller's CSR
    found = [e for e in range(E) if SIZES[e]]
    step = rows * rb
    g = K.expert_ptrs([(0, 0, ptr[0] + e * step) if down else (ptr[0] + e * step, ptr[1] + e * step, 0) for e in found])
    pairs = np.concatenate([(i := np.flatnonzero(ids.reshape(-1) == e)) // n_used << 4 | i % n_used for e in found])
    starts = np.concatenate([[0], np.cumsum([SIZES[e] for e in found])]).astype(np.uint32)
    dg, ds, dp = up(g), up(starts), up(pairs.astype(np.uint32))
    got = zeros_f32((T * n_used, rows))
    if down:
        K.moe_down_grouped(got, dg, ds, dp, d_xq, cols, rows, n_used, len(found), rb, quant)
    else:
        K.moe_pair_swiglu_grouped(got, dg, ds, dp, d_w, d_xq, cols, rows, n_used, len(found), rb, quant, 0)
    csr = down_np(got)
    check_grouped(quant, mats, ids, xq, wts, csr, down, cols, "csr")
    assert not csr[np.flatnonzero(ids.reshape(-1) == -1)].any()  # unlisted rows stay untouched
    # the router's ids
    first = list(dict.fromkeys(int(e) for e in ids.reshape(-1) if e >= 0))
    active = np.zeros(2 + E, np.uint32)
    active[:2 + len(first)] = [len(first), int((ids == -1).sum())] + first
    bank = (K.ExpertBank(None, None, ptr[0], None, None, None, 0, 0, step, 0, 0, 0) if down else
            K.ExpertBank(ptr[0], ptr[1], None, None, None, None, step, step, 0, 0, 0, 0))
    got = torch.full((T * n_used, rows), float("nan"), dtype=torch.float32, device=dev)
    d_ids, d_act = up(ids), up(active)
    if down:
        K.moe_down_experts(got, d_ids, d_act, d_xq, bank, E, [], T, n_used, cols, rows, rb, quant)
    else:
        K.moe_pair_swiglu_experts(got, d_ids, d_act, d_w, d_xq, bank, E, [], T, n_used, cols, rows, rb, quant, 0)
    exp = down_np(got)
    check_grouped(quant, mats, ids, xq, wts, exp, down, cols, "experts")
    assert not exp[np.flatnonzero(ids.reshape(-1) == -1)].any()  # NULL slots: rows of 0
    assert np.array_equal(csr, exp)  # both on the tile: the same sums


def test_tile_shared_slot(dev):
    """Few pairs per routed expert, every token in a shared slot: the routed
    groups on the 16-row kernel, the shared one on the tile."""
    quant, hidden, ffn, T, E, k = QUANT_Q4_K, 512, 96, 40, 64, 2
    rng = np.random.default_rng(4)
    mats, _, xq = grouped_case(quant, hidden, ffn, [0] * (E + 1), 1, rng, False)
    xq = oracle.quantize_q8_k(rng.standard_normal((T, hidden)).astype(np.float32) * 1e-2)
    ids = np.stack([rng.choice(E, k, replace=False) for _ in range(T)]).astype(np.int32)
    rb, first = row_bytes(quant, hidden), list(dict.fromkeys(int(e) for e in ids.reshape(-1)))
    active = np.zeros(2 + E, np.uint32)
    active[:2 + len(first)] = [len(first), 0] + first
    wts = np.concatenate([rng.uniform(0.1, 1, (T, k)), np.ones((T, 1))], 1).astype(np.float32)
    dm, step = [up(m) for m in mats], ffn * rb
    bank = K.ExpertBank(dm[0].data_ptr(), dm[1].data_ptr(), None, None, None, None, step, step, 0, 0, 0, 0)
    shared = [(dm[0].data_ptr() + E * step, dm[1].data_ptr() + E * step, 0)]
    got = torch.full((T * (k + 1), ffn), float("nan"), dtype=torch.float32, device=dev)
    K.moe_pair_swiglu_experts(got, up(ids), up(active), torch.from_numpy(wts).to(dev), up(xq), bank, E, shared, T, k,
                              hidden, ffn, rb, quant, 0)
    all_ids = np.concatenate([ids, np.full((T, 1), E, np.int32)], 1)
    check_grouped(quant, mats, all_ids, xq, wts, down_np(got), False, hidden, "shared")
