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
