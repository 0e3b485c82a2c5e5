"""The tile shapes for up to a round of tiles (bf16: 32x64, 64x64 with eight wavefronts, 64x128 with two K groups): sizes at which
the size rule picks each, with border tiles in both directions and contractions of one step, of a whole number of steps, and of one
element more or less, at the bars of the other tile shapes."""
import pytest

import test_gpu_gemm_tile as tiles
from util import DTYPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,m,k", [(505, 776, 1001), (512, 768, 768), (449, 760, 257), (481, 768, 2305), (500, 770, 511),   # 32x64
                                   (320, 2310, 770), (1000, 768, 129), (1024, 768, 128), (520, 770, 40), (970, 776, 3071),  # 64x64
                                   (1500, 768, 768), (700, 2310, 771), (1536, 760, 2305), (513, 3080, 257), (1409, 776, 1023)])  # 64x128
@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
def test_tiles_of_one_round(mt, dtype, n, m, k, layout):
    tiles.test_tile_shapes(mt, dtype, n, m, k, layout)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,m,k", [(505, 776, 769), (320, 2312, 768), (970, 776, 257), (1500, 768, 770), (513, 3072, 768)])
def test_multiplied_tiles_of_one_round(mt, dtype, n, m, k):
    tiles.test_tile_multiply_epilogue(mt, dtype, n, m, k)
