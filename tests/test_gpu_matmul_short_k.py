"""float32 products on both sides of the K up to which the small blocks are preferred."""

import numpy as np
import pytest

from helpers import encode, pair
from raven_amd import dtype as dt
from test_gpu_matmul import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,path", [(32, "gemm_tile_64x64"), (64, "gemm_tile_64x64"), (96, "gemm_tile_128x64")])
def test_block_shape_of_a_short_k(hip, oracle, k, path):
    rng = np.random.default_rng(k)
    d, b, m, n = dt.float32, 32, 288, 784
    w, y = encode(rng.standard_normal((k, m)), d, oracle), encode(rng.standard_normal((b, k, n)), d, oracle)
    hw = pair(w, d, hip, oracle, lambda B, t: B.expand(B.reshape(B.permute(t, (1, 0)), (1, m, k)), (b, m, k)))[0]
    check(hip, oracle, d, hw, pair(y, d, hip, oracle)[0], np.broadcast_to(w.T, (b, m, k)), y, f"{m}x{k}x{n}")
    assert hip.last_path() == path
