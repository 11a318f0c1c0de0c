"""Which kernel a grouped expert stage runs on, and that its rows do not show it:
the 16-row kernel (csrc/mmq.hip), the wide tile (csrc/tile_moe.hip) and the lane
kernels (csrc/moe.hip) take a stage by the size of its groups, so every case here
puts the same pairs on two sides of a choice or checks one side on the oracle."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from pulsar_amd import formats as fm
from pulsar_amd import kernels as K
from pulsar_amd import runtime, synth
from pulsar_amd.formats import QUANT_IQ2_XXS, QUANT_IQ4_XS, QUANT_Q2_K, QUANT_Q3_K, QUANT_Q4_K, QUANT_Q5_K, QUANT_Q6_K, row_bytes
from tests.gpu_util import down as down_np
from tests.gpu_util import assert_rows_close, up, zeros_f32
from tests.test_gpu_tile import FORMATS, SIZES, check_grouped, edge_rows, grouped_case, rows_want

pytestmark = pytest.mark.gpu
ROW16 = [QUANT_Q2_K, QUANT_IQ2_XXS, QUANT_Q4_K, QUANT_Q5_K, QUANT_Q6_K]  # formats of the 16-row kernel and the tile


class Stage:
    """One grouped stage over groups of the given sizes (expert e: sizes[e]
    pairs), callable from a caller's CSR and from the router's ids."""

    def __init__(self, dev, quant, down, sizes, hidden=768, ffn=330, n_used=3, seed=0):
        rng = np.random.default_rng(seed + 2 * quant + down)
        self.dev, self.quant, self.down, self.sizes, self.n_used = dev, quant, down, list(sizes), n_used
        self.rows, self.cols = (hidden, ffn) if down else (ffn, hidden)
        self.mats, self.ids, self.xq = grouped_case(quant, hidden, ffn, self.sizes, n_used, rng, down)
        self.T, self.E, self.rb = self.ids.shape[0], len(self.sizes), row_bytes(quant, self.cols)
        self.wts = rng.uniform(0.1, 1.0, (self.T, n_used)).astype(np.float32)
        self.d_mats, self.d_xq, self.d_w = [up(m) for m in self.mats], up(self.xq), torch.from_numpy(self.wts).to(dev)
        self.step = self.rows * self.rb

    def entry(self, e):
        p = [m.data_ptr() + e * self.step for m in self.d_mats]
        return (0, 0, p[0]) if self.down else (p[0], p[1], 0)

    def csr_arrays(self, order=None, pad=0, skip=0):
        """gptrs, starts, pairs of the experts in `order` (all; -1: an empty NULL
        group), then `pad` empty NULL groups; the listed pairs start at `skip`."""
        order = list(range(self.E)) if order is None else list(order)
        order += [-1] * pad
        flat = self.ids.reshape(-1)
        lists = [np.flatnonzero(flat == e) if e >= 0 else np.zeros(0, np.int64) for e in order]
        g = K.expert_ptrs([self.entry(e) if e >= 0 else (0, 0, 0) for e in order])
        i = np.concatenate(lists)
        pairs = np.concatenate([np.zeros(skip, np.int64), i // self.n_used << 4 | i % self.n_used]).astype(np.uint32)
        starts = (skip + np.concatenate([[0], np.cumsum([len(v) for v in lists])])).astype(np.uint32)
        return g, starts, pairs

    def queue_csr(self, dev_arrays, n_group, out, xq=None):
        g, starts, pairs = dev_arrays
        xq = self.d_xq if xq is None else xq
        if self.down:
            K.moe_down_grouped(out, g, starts, pairs, xq, self.cols, self.rows, self.n_used, n_group, self.rb, self.quant)
        else:
            K.moe_pair_swiglu_grouped(out, g, starts, pairs, self.d_w, xq, self.cols, self.rows, self.n_used, n_group,
                                      self.rb, self.quant, 0)

    def zeros(self):
        return torch.zeros((self.T * self.n_used, self.rows), dtype=torch.float32, device=self.dev)

    def run_csr(self, arrays, xq=None):
        out, dev_arrays = self.zeros(), [up(a) for a in arrays]
        torch.cuda.synchronize()
        self.queue_csr(dev_arrays, len(arrays[1]) - 1, out, xq)
        return down_np(out)

    def run_experts(self, xq=None):
        ids = self.ids.reshape(-1)
        first = list(dict.fromkeys(int(e) for e in ids if e >= 0))
        active = np.zeros(2 + self.E, np.uint32)
        active[:2 + len(first)] = [len(first), int((ids == -1).sum())] + first
        p = [m.data_ptr() for m in self.d_mats]
        bank = (K.ExpertBank(None, None, p[0], None, None, None, 0, 0, self.step, 0, 0, 0) if self.down else
                K.ExpertBank(p[0], p[1], None, None, None, None, self.step, self.step, 0, 0, 0, 0))
        out = torch.full((self.T * self.n_used, self.rows), float("nan"), dtype=torch.float32, device=self.dev)
        d_ids, d_act, xq = up(self.ids), up(active), self.d_xq if xq is None else xq
        if self.down:
            K.moe_down_experts(out, d_ids, d_act, xq, bank, self.E, [], self.T, self.n_used, self.cols, self.rows,
                               self.rb, self.quant)
        else:
            K.moe_pair_swiglu_experts(out, d_ids, d_act, self.d_w, xq, bank, self.E, [], self.T, self.n_used,
                                      self.cols, self.rows, self.rb, self.quant, 0)
        return down_np(out)

    def check(self, got, what):
        check_grouped(self.quant, self.mats, self.ids, self.xq, self.wts, got, self.down, self.cols, what)


@pytest.mark.parametrize("down", [False, True])
@pytest.mark.parametrize("quant", ROW16, ids=lambda q: fm.NAMES[q])
def test_rows_equal_across_kernels(dev, quant, down):
    """The same groups from a CSR whose padding makes their mean short (the
    16-row kernel) and from the router's ids (the tile): bit for bit equal."""
    s = Stage(dev, quant, down, SIZES, *((330, 768) if down else (768, 330)))
    short, tile = s.run_csr(s.csr_arrays(pad=400)), s.run_experts()
    s.check(short, "16-row")
    assert np.array_equal(short.view(np.uint32), tile.view(np.uint32))
    assert np.array_equal(s.run_csr(s.csr_arrays()).view(np.uint32), tile.view(np.uint32))


def shifted(a, off, dev):
    """A device copy of the bytes of `a` that starts `off` bytes past a 256-byte
    boundary."""
    t = torch.zeros(a.size + 256, dtype=torch.uint8, device=dev)[off:off + a.size]
    t.copy_(torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)))
    assert t.data_ptr() % 4 == off % 4
    return t


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("quant", FORMATS, ids=lambda q: fm.NAMES[q])
def test_q8_rows_at_any_byte(dev, quant, off):
    """q8_K rows that do not start on a dword, which the tile's copies to LDS
    cannot read: chunks and groups long enough for the tile, on the oracle."""
    rows, n_tok, n = 4129, 130, 768
    w = synth.quant_matrix(quant, rows, n, synth.rng_for(off, "shift"))
    xq = oracle.quantize_q8_k(np.random.default_rng(off).standard_normal((n_tok, n)).astype(np.float32))
    out = zeros_f32((n_tok, rows))
    K.matmul_kq(out, up(w), shifted(xq, off, dev), n, rows, n_tok, row_bytes(quant, n), quant)
    at = edge_rows(rows)
    want, _, bound = rows_want(quant, np.ascontiguousarray(w[at]), row_bytes(quant, n), xq, n, n_tok)
    assert_rows_close(down_np(out)[:, at], want, bound, f"{fm.NAMES[quant]} +{off}")
    for down in (False, True):
        s = Stage(dev, quant, down, [70, 1, 0, 129], 256, 256)
        x = shifted(s.xq, off, dev)
        s.check(s.run_csr(s.csr_arrays(), xq=x), "csr")
        s.check(s.run_experts(xq=x), "experts")


class KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint * 3), ("args", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def launches(fn):
    """The kernel nodes of a graph of fn's launches (recorded, not run)."""
    hip, graph, n = runtime._hip(), ctypes.c_void_p(), ctypes.c_size_t()
    runtime._check(hip.hipStreamBeginCapture(runtime.STREAM_PER_THREAD, runtime.CAPTURE_THREAD_LOCAL), "begin")
    try:
        fn()
    finally:
        runtime._check(hip.hipStreamEndCapture(runtime.STREAM_PER_THREAD, ctypes.byref(graph)), "end")
    hip.hipGraphGetNodes.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_size_t)]
    hip.hipGraphKernelNodeGetParams.argtypes = [ctypes.c_void_p, ctypes.POINTER(KernelNode)]
    runtime._check(hip.hipGraphGetNodes(graph, None, ctypes.byref(n)), "nodes")
    nodes = (ctypes.c_void_p * n.value)()
    runtime._check(hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)), "nodes")
    out = []
    for node in nodes:
        k = KernelNode()
        runtime._check(hip.hipGraphKernelNodeGetParams(node, ctypes.byref(k)), "node")
        out.append(k)
    hip.hipGraphDestroy(graph)
    return out


# formats and row lengths (14336 values do not fit the 16-row kernel) whose
# short groups run on the lane kernels; sizes whose mean is on one side of the
# tile's bound for the CSR and for the router's ids alike
LANE_TILE = [(QUANT_Q3_K, False, 512), (QUANT_Q3_K, True, 768), (QUANT_IQ4_XS, False, 768), (QUANT_IQ4_XS, True, 512),
             (QUANT_Q4_K, False, 14336), (QUANT_Q2_K, True, 14336), (QUANT_Q6_K, True, 14336)]


@pytest.mark.parametrize("long", [False, True])
@pytest.mark.parametrize("quant,down,cols", LANE_TILE, ids=lambda v: str(v))
def test_lane_or_tile_by_the_mean(dev, quant, down, cols, long):
    """A CSR of short groups runs on the lane kernels, of long ones on the tile,
    as the router's ids do: both on the oracle, and equal bit for bit."""
    sizes = [40, 33, 50] if long else [1] * 40
    s = Stage(dev, quant, down, sizes, *((70, cols) if down else (cols, 70)), n_used=1)
    csr, ids = s.run_csr(s.csr_arrays()), s.run_experts()
    s.check(csr, "csr")
    s.check(ids, "experts")
    assert np.array_equal(csr.view(np.uint32), ids.view(np.uint32))


@pytest.mark.parametrize("down", [False, True])
@pytest.mark.parametrize("quant", FORMATS, ids=lambda q: fm.NAMES[q])
def test_short_csr_is_one_launch(dev, quant, down):
    """A CSR that cannot list enough pairs for the tile (here 40 in 60 groups)
    takes one launch; with the capacity unknown, as through a raw address, or
    with room for long groups it takes two, and the rows are the same."""
    s = Stage(dev, quant, down, [1] * 40, *((70, 512) if down else (512, 70)))
    g, starts, pairs = (up(a) for a in s.csr_arrays(pad=20))
    roomy = torch.zeros(4 * 4096, dtype=torch.uint8, device=dev)
    roomy[:pairs.numel()] = pairs

    def stage(pairs):
        out = s.zeros()
        torch.cuda.synchronize()

        def call():
            s.queue_csr((g, starts, pairs), 60, out)

        n = len(launches(call))
        call()
        return n, down_np(out).view(np.uint32)

    (n1, a), (n2, b), (n3, c) = stage(pairs), stage(pairs.data_ptr()), stage(roomy)
    assert (n1, n2, n3) == (1, 2, 2)
    assert np.array_equal(a, b) and np.array_equal(a, c)
    s.check(a.view(np.float32), "csr")


@pytest.mark.parametrize("down", [False, True])
def test_few_long_groups_fill_the_chip(dev, down):
    """One group of many pair tiles is spread over as many blocks as many
    groups are: the tiles count, not the groups."""
    s = Stage(dev, QUANT_Q4_K, down, [1500], *((330, 512) if down else (512, 330)))
    dev_arrays = [up(a) for a in s.csr_arrays()]
    out = s.zeros()
    torch.cuda.synchronize()
    assert launches(lambda: s.queue_csr(dev_arrays, 1, out))[-1].grid[0] == 512
    s.check(s.run_csr(s.csr_arrays()), "csr")


# (format, down, experts, rows, cols, tokens, top): stages of which the 16-row
# kernel was timed faster than the tile (at the left of the line between the
# two, by format, row length and pairs per expert), and slower
ON_ROW16 = [(QUANT_IQ2_XXS, False, 32, 2816, 2816, 48, 4), (QUANT_IQ2_XXS, False, 8, 14336, 4096, 24, 2),
            (QUANT_Q2_K, False, 16, 6400, 4096, 40, 2), (QUANT_Q2_K, False, 32, 2816, 2816, 32, 4),
            (QUANT_Q5_K, False, 32, 2816, 2816, 40, 4), (QUANT_IQ2_XXS, False, 128, 768, 2048, 96, 8),
            (QUANT_IQ2_XXS, True, 128, 2048, 768, 256, 8), (QUANT_Q6_K, True, 128, 2048, 768, 192, 8)]
ON_TILE = [(QUANT_IQ2_XXS, False, 32, 2816, 2816, 80, 4), (QUANT_Q2_K, False, 128, 1536, 4096, 80, 8),
           (QUANT_Q4_K, False, 128, 768, 2048, 96, 8), (QUANT_Q5_K, False, 32, 2816, 2816, 80, 4),
           (QUANT_Q6_K, True, 128, 2048, 768, 256, 8), (QUANT_Q6_K, True, 8, 4096, 14336, 24, 2)]


@pytest.mark.parametrize("stage", ON_ROW16 + ON_TILE, ids=lambda s: "-".join(map(str, s)))
def test_choice_by_measured_crossover(dev, stage):
    """The kernel a stage of the router's ids is recorded on (nothing runs):
    the tile's only dynamic LDS is the pair list, 4 bytes a routed pair."""
    quant, down, E, rows, cols, T, k = stage
    bank = K.ExpertBank(256, 256, 256, None, None, None, 0, 0, 0, 0, 0, 0)  # addresses are not read
    buf = torch.zeros(256, dtype=torch.uint8, device=dev)

    def call():
        if down:
            K.moe_down_experts(buf, buf, buf, buf, bank, E, [], T, k, cols, rows, row_bytes(quant, cols), quant)
        else:
            K.moe_pair_swiglu_experts(buf, buf, buf, buf, buf, bank, E, [], T, k, cols, rows, row_bytes(quant, cols),
                                      quant, 0)

    nodes = launches(call)
    assert len(nodes) == 1
    assert (nodes[0].shared == 4 * T * k) == (stage in ON_TILE)


@pytest.mark.parametrize("stage", [
    # format, down, groups, rows, cols, the most pairs per group short of the line and the least past it
    (QUANT_Q4_K, False, 128, 768, 2048, 7, 8), (QUANT_Q2_K, False, 128, 1536, 4096, 6, 8),
    (QUANT_IQ2_XXS, False, 128, 1536, 4096, 7, 9), (QUANT_Q6_K, True, 128, 2048, 768, 24, 28),
    (QUANT_Q4_K, True, 256, 2048, 512, 12, 16), (QUANT_IQ4_XS, True, 256, 2048, 512, 2, 3)],
    ids=lambda s: "-".join(map(str, s)))
def test_csr_choice_by_measured_crossover(dev, stage):
    """A CSR that can hold groups past the line takes the tile's launch too, one
    short of it does not (recorded, not run)."""
    quant, down, groups, rows, cols, under, over = stage
    buf = torch.zeros(256, dtype=torch.uint8, device=dev)
    for per_group, want in ((under, 1), (over, 2)):
        pairs = torch.zeros(per_group * groups, dtype=torch.int32, device=dev)

        def call():
            if down:
                K.moe_down_grouped(buf, buf, buf, pairs, buf, cols, rows, 8, groups, row_bytes(quant, cols), quant)
            else:
                K.moe_pair_swiglu_grouped(buf, buf, buf, pairs, buf, buf, cols, rows, 8, groups, row_bytes(quant, cols),
                                          quant, 0)

        assert len(launches(call)) == want


# ------------------------------------------ the tile's branches, on the oracle

@pytest.mark.parametrize("act", [fm.ACT_SILU, fm.ACT_SWIGLU_OAI])
@pytest.mark.parametrize("quant", [QUANT_Q4_K, QUANT_Q2_K, QUANT_Q6_K, QUANT_IQ4_XS], ids=lambda q: fm.NAMES[q])
def test_tile_biases_and_activation(dev, quant, act):
    """Gate and up biases (one expert without) and both activations on the tile,
    from both sources, against the oracle's dots."""
    sizes = [70, 33, 40]
    s = Stage(dev, quant, False, sizes, 512, 200)
    rng = np.random.default_rng(act)
    bias = [rng.standard_normal((s.E, s.rows)).astype(np.float32) for _ in range(2)]
    d_bias = [torch.from_numpy(b).to(dev) for b in bias]
    order = list(range(s.E))
    _, starts, pairs = s.csr_arrays(order)
    g = K.expert_ptrs([s.entry(e) + tuple(b.data_ptr() + 4 * e * s.rows if e != 1 else 0 for b in d_bias)
                       for e in order])
    csr = s.zeros()
    K.moe_pair_swiglu_grouped(csr, up(g), up(starts), up(pairs), s.d_w, s.d_xq, s.cols, s.rows, s.n_used, s.E, s.rb,
                              quant, act)
    got = {"csr": down_np(csr)}
    p = [m.data_ptr() for m in s.d_mats]
    active = np.array([s.E, int((s.ids == -1).sum())] + order, np.uint32)
    bank = K.ExpertBank(p[0], p[1], None, d_bias[0].data_ptr(), d_bias[1].data_ptr(), None, s.step, s.step, 0, s.rows,
                        s.rows, 0)
    exp = s.zeros()
    K.moe_pair_swiglu_experts(exp, up(s.ids), up(active), s.d_w, s.d_xq, bank, s.E, [], s.T, s.n_used, s.cols, s.rows,
                              s.rb, quant, act)
    got["experts"] = down_np(exp)
    flat = s.ids.reshape(-1)
    for e in order:
        at = np.flatnonzero(flat == e)
        (gv, _, bg), (uv, _, bu) = (rows_want(quant, m[e], s.rb, s.xq[at // s.n_used], s.cols, at.size) for m in s.mats)
        gv, uv, bg, bu = (v.astype(np.float64) for v in (gv, uv, 1e-5 * bg, 1e-5 * bu))
        w = s.wts.reshape(-1)[at].astype(np.float64)[:, None]
        for who, rows in got.items():
            g0, u0, eg, eu = gv, uv, bg, bu
            if e != 1 or who == "experts":  # the bank gives every expert its biases
                g0, u0 = gv + bias[0][e], uv + bias[1][e]
                eg, eu = bg + 2.0**-24 * np.abs(g0), bu + 2.0**-24 * np.abs(u0)
            if act == fm.ACT_SWIGLU_OAI:  # the clamps spread no error; sigmoid sharpened by 1.702
                g1 = np.minimum(g0, 7.0)
                a, f = g1 / (1 + np.exp(-1.702 * g1)), np.clip(u0, -7, 7) + 1
            else:
                a, f = g0 / (1 + np.exp(-g0)), u0
            # |(g sigmoid(k g))'| <= 1.1 for either k; exp, division and products: 1e-6
            bound = w * (1.1 * eg * (np.abs(f) + eu) + np.abs(a) * eu) + 1e-6 * np.abs(a * f) * w + 1e-30
            err = np.abs(rows[at] - a * f * w)
            assert (err <= bound).all(), (who, e, float((err / bound).max()))


@pytest.mark.parametrize("down", [False, True])
@pytest.mark.parametrize("quant", [QUANT_Q4_K, QUANT_Q6_K, QUANT_Q3_K], ids=lambda q: fm.NAMES[q])
def test_tile_csr_forms(dev, quant, down):
    """CSRs the device-built ones never are: pairs that start past the first
    entry, empty groups between full ones, a group with pairs and NULL pointers
    (its rows stay untouched)."""
    sizes = [40, 0, 65, 1, 0, 130]
    s = Stage(dev, quant, down, sizes, *((200, 512) if down else (512, 200)))
    whole = s.run_csr(s.csr_arrays())
    s.check(whole, "csr")
    order = [-1, 0, 1, -1, -1, 2, 3, 4, 5, -1]
    assert np.array_equal(s.run_csr(s.csr_arrays(order, skip=37)).view(np.uint32), whole.view(np.uint32))
    g, starts, pairs = s.csr_arrays()
    g[2] = 0
    got, null = s.run_csr((g, starts, pairs)), s.ids.reshape(-1) == 2
    assert not got[null].any()
    assert np.array_equal(got[~null].view(np.uint32), whole[~null].view(np.uint32))


@pytest.mark.parametrize("quant", [QUANT_Q4_K, QUANT_Q3_K], ids=lambda q: fm.NAMES[q])
@pytest.mark.parametrize("groups", [1023, 1024, 1025])
def test_csr_of_many_groups(dev, quant, groups):
    """The tile counts the tiles of up to 1024 groups; a CSR of more stays on the
    kernels without that limit. 12 pairs per group, 8 matrices."""
    s = Stage(dev, quant, False, [12] * 8, 512, 64)
    order = np.arange(groups) % s.E
    g, starts, pairs = s.csr_arrays()
    lists = [pairs[starts[e]:starts[e + 1]] for e in range(s.E)]
    arrays = (g[order], (12 * np.arange(groups + 1)).astype(np.uint32), np.concatenate([lists[e] for e in order]))
    out, dev_arrays = s.zeros(), [up(a) for a in arrays]
    n = len(launches(lambda: s.queue_csr(dev_arrays, groups, out)))
    assert n == (1 if groups > 1024 else 2)
    s.check(s.run_csr(arrays), "csr")


def test_skewed_groups_on_the_16_row_kernel(dev):
    """One long group among many single pairs: the mean keeps the stage on the
    16-row kernel, which walks the long one in several pair tiles; the same rows
    as where that group is alone and long enough for the tile."""
    for quant in ROW16:
        for down in (False, True):
            s = Stage(dev, quant, down, [150] + [1] * 199, *((77, 512) if down else (512, 77)), n_used=2)
            both = s.run_csr(s.csr_arrays())
            s.check(both, "skewed")
            alone, at = s.run_csr(s.csr_arrays([0])), s.ids.reshape(-1) == 0
            assert np.array_equal(both[at].view(np.uint32), alone[at].view(np.uint32)), (fm.NAMES[quant], down)


@pytest.mark.parametrize("quant", [QUANT_Q4_K, QUANT_Q2_K, QUANT_Q6_K], ids=lambda q: fm.NAMES[q])
@pytest.mark.parametrize("n_tok", [33, 128])
def test_shared_slot_equal_from_both_sources(dev, quant, n_tok):
    """Few pairs per routed expert and a shared slot of every token: from the
    router's ids the shared group is a launch of its own on the tile (gate / up
    from 33 tokens, down from 100), in a CSR one group among the others."""
    E, k = 256, 2
    for down in (False, True):
        sizes = [1] * E + [n_tok]
        s = Stage(dev, quant, down, sizes, *((140, 512) if down else (512, 140)), n_used=3)
        rng = np.random.default_rng(n_tok)
        ids = np.stack([np.append(rng.choice(E, k, replace=False), E) for _ in range(n_tok)]).astype(np.int32)
        s.ids, s.T = ids, n_tok
        s.xq = oracle.quantize_q8_k(rng.standard_normal((n_tok * (3 if down else 1), s.cols)).astype(np.float32) * 1e-2)
        s.wts = np.concatenate([rng.uniform(0.1, 1, (n_tok, k)), np.ones((n_tok, 1))], 1).astype(np.float32)
        s.d_xq, s.d_w = up(s.xq), torch.from_numpy(s.wts).to(dev)
        csr = s.run_csr(s.csr_arrays())
        s.check(csr, "csr")
        first = list(dict.fromkeys(int(e) for e in ids[:, :k].reshape(-1)))
        active = np.zeros(2 + E, np.uint32)
        active[:2 + len(first)] = [len(first), 0] + first
        p = [m.data_ptr() for m in s.d_mats]
        out, args = s.zeros(), (up(np.ascontiguousarray(ids[:, :k])), up(active))
        if down:
            bank = K.ExpertBank(None, None, p[0], None, None, None, 0, 0, s.step, 0, 0, 0)
            call = lambda: K.moe_down_experts(out, *args, s.d_xq, bank, E, [s.entry(E)], n_tok, k, s.cols, s.rows, s.rb,
                                              quant)
        else:
            bank = K.ExpertBank(p[0], p[1], None, None, None, None, s.step, s.step, 0, 0, 0, 0)
            call = lambda: K.moe_pair_swiglu_experts(out, *args, s.d_w, s.d_xq, bank, E, [s.entry(E)], n_tok, k, s.cols,
                                                     s.rows, s.rb, quant, 0)
        assert len(launches(call)) == (2 if not down or n_tok >= 100 else 1)
        call()
        assert np.array_equal(down_np(out).view(np.uint32), csr.view(np.uint32)), down


@pytest.mark.parametrize("down", [False, True])
def test_tile_of_2048_ids(dev, down):
    """The most ids a block scans: 2048, a quarter to each wave, 8 strips of 64."""
    s = Stage(dev, QUANT_Q4_K, down, [300, 700, 1, 450, 585], *((70, 512) if down else (512, 70)), n_used=4)
    assert s.ids.size == 2048  # 12 of them route nowhere
    got = s.run_experts()
    s.check(got, "experts")
    assert not got[s.ids.reshape(-1) == -1].any()


@pytest.mark.parametrize("quant,down", [(QUANT_Q4_K, False), (QUANT_Q6_K, True), (QUANT_Q3_K, False)])
def test_csr_graph_follows_the_group_sizes(dev, quant, down):
    """A CSR stage captured once, its arrays replaced between replays: short,
    long, short and unevenly long groups take their kernel inside the same graph,
    and every replay equals an eager run."""
    E = 24
    s = Stage(dev, quant, down, [40] * E, *((140, 512) if down else (512, 140)))
    flat = s.ids.reshape(-1)
    cap, out = up(np.zeros(flat.size, np.uint32)), s.zeros()
    g, starts = up(s.csr_arrays()[0]), up(np.zeros(E + 1, np.uint32))
    call = lambda: s.queue_csr((g, starts, cap), E, out)
    graph = runtime.Graph.capture(call)
    for per in ([1] * E, [40] * E, [2] * E, [40] * 3 + [1] * (E - 3), [0] * (E - 1) + [40], [40] * E):
        lists = [np.flatnonzero(flat == e)[:n] for e, n in enumerate(per)]
        i = np.concatenate(lists)
        pairs = np.zeros(flat.size, np.uint32)
        pairs[:i.size] = i // s.n_used << 4 | i % s.n_used
        cap.copy_(up(pairs))
        starts.copy_(up(np.concatenate([[0], np.cumsum([len(v) for v in lists])]).astype(np.uint32)))
        out.zero_()
        torch.cuda.synchronize()
        graph.launch()
        runtime.sync()
        replay = down_np(out).copy()
        out.zero_()
        torch.cuda.synchronize()
        call()
        runtime.sync()
        assert np.array_equal(replay.view(np.uint32), down_np(out).view(np.uint32)), per
        listed = np.zeros(flat.size, bool)
        listed[i] = True
        assert replay[listed].any(1).all() and not replay[~listed].any()
