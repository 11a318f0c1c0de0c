"""Which kernel a dense prompt chunk is recorded on: the wide tile (csrc/tile.hip)
or the 16-row and lane kernels, by format, rows, columns and tokens, at shapes
where either was timed faster."""
import pytest
import torch

from pulsar_amd import kernels as K
from pulsar_amd.formats import (QUANT_IQ2_XXS, QUANT_IQ4_XS, QUANT_Q2_K, QUANT_Q3_K, QUANT_Q4_K, QUANT_Q5_K, QUANT_Q6_K,
                                row_bytes)
from tests.test_gpu_grouped_choice import launches

pytestmark = pytest.mark.gpu

# (format, rows, columns, tokens)
OTHER = [(QUANT_IQ4_XS, 1024, 256, 64), (QUANT_IQ4_XS, 2048, 512, 24), (QUANT_IQ2_XXS, 4096, 512, 6),
         (QUANT_IQ2_XXS, 4096, 8192, 5), (QUANT_IQ2_XXS, 1024, 1536, 32), (QUANT_Q2_K, 2048, 512, 13),
         (QUANT_Q3_K, 1024, 512, 32), (QUANT_Q4_K, 8192, 512, 64), (QUANT_Q5_K, 8192, 512, 64),
         (QUANT_Q5_K, 14336, 256, 32), (QUANT_Q5_K, 11008, 8192, 64), (QUANT_Q6_K, 3000, 2048, 100)]
TILE = [(QUANT_IQ4_XS, 4096, 512, 17), (QUANT_IQ2_XXS, 4096, 6144, 8), (QUANT_IQ2_XXS, 2048, 4096, 17),
        (QUANT_Q2_K, 4096, 512, 17), (QUANT_Q3_K, 2048, 2048, 16), (QUANT_Q4_K, 4096, 4096, 33),
        (QUANT_Q5_K, 4096, 4096, 64), (QUANT_Q5_K, 14336, 4096, 48), (QUANT_Q6_K, 14336, 4096, 64)]


def tile_grids(rows, tokens):
    """The grids of the tile's four shapes: rows x tokens of a block, padded to
    the 8 XCDs."""
    return {(-(-rows // r) * -(-tokens // t) + 7) & ~7 for r, t in ((32, 32), (64, 64), (128, 64), (128, 128))}


@pytest.mark.parametrize("shape", OTHER + TILE, ids=lambda s: "-".join(map(str, s)))
def test_choice_by_measured_crossover(dev, shape):
    quant, rows, cols, tokens = shape
    buf = torch.zeros(256, dtype=torch.uint8, device=dev)  # recorded, not run
    nodes = launches(lambda: K.matmul_kq(buf, buf, buf, cols, rows, tokens, row_bytes(quant, cols), quant))
    assert len(nodes) == 1
    grid = tuple(nodes[0].grid)
    assert (grid[1:] == (1, 1) and grid[0] in tile_grids(rows, tokens)) == (shape in TILE), grid
