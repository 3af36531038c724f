"""GEMMs on tiles of 256 columns: every number of rows that a workgroup takes, with the last row tile and the last columns not filled and as
many stages of k as the ring holds and more.  References and bounds are those of the tests of the other tiles."""
import pytest

import test_gpu_decoder_sizes as floats
import test_gpu_gemm_tiles as ints
from test_gpu_prefill import fx  # noqa: F401

pytestmark = pytest.mark.gpu

# rows of a workgroup: rows and columns of a product
FLOAT = {128: (300, 12284), 160: (1299, 12284), 192: (1632, 12288), 224: (2076, 6140), 256: (1151, 12284)}
FLOAT_K = [320, 576]
INT = {(128, 1152): (300, 12284), (160, 1152): (1558, 6144), (192, 1152): (1632, 6140), (224, 384): (2076, 6144), (224, 1152): (1928, 6140),
       (256, 384): (1151, 12284), (256, 1152): (1151, 12288)}


@pytest.mark.parametrize("k", FLOAT_K)
@pytest.mark.parametrize("split,glu", [("all", 0), ("all", 1), ("half", 2), ("none", 0)])
@pytest.mark.parametrize("rows", FLOAT)
def test_rows_bfloat16(rows, split, glu, k):
    m, n = FLOAT[rows]
    floats.test_gemm_tiles(m, n, {"all": n, "half": n // 512 * 256 + 64, "none": 0}[split], glu, k, "bfloat16")


@pytest.mark.parametrize("rows,k", INT)
def test_rows_int8(fx, oracle, rows, k):  # noqa: F811
    m, n = INT[rows, k]
    ints.test_tiles(fx, oracle, m, k, n)
    ints.test_half_line_tiles_with_the_gated_unit(fx, m, k, n)
