"""A few rows times a 16-bit matrix in memory order (gemm_strip.hip), at the edges of its tiles, its steps
and its shares of K; the fused linear, alone and in a group, has the bits of the calls that it stands for."""

import numpy as np
import pytest

from helpers import decode, encode, pair, same_bits
from raven_amd import dtype as dt
from raven_amd.kaun_gpt2 import Config, Gpt2, Linear
from raven_amd.nx_backend import logical
from raven_amd.nx_frontend import Nx
from test_gpu_defer import deferred
from test_gpu_matmul import check

pytestmark = pytest.mark.gpu
HALVES = [dt.bfloat16, dt.float16]


@pytest.mark.parametrize("d", HALVES, ids=lambda d: d.name)
@pytest.mark.parametrize("m,k,n,path", [
    (1, 512, 512, "gemm_strip"), (16, 448, 515, "gemm_strip"), (17, 640, 520, "gemm_strip"),  # one row tile and beside
    (48, 768, 768, "gemm_strip"), (300, 704, 577, "gemm_strip"), (384, 512, 1024, "gemm_strip"),  # 16, 32 and 64 rows a tile
    (5, 256, 2049, "gemm_strip"), (33, 287, 513, "gemm_strip"), (63, 511, 66, "gemm_strip"), (64, 2001, 8190, "gemm_strip"),  # K off a step
    (33, 5300, 500, "gemm_strip"), (16, 11109, 314, "gemm_strip"), (3, 4700, 571, "gemm_strip"),  # K cut among blocks
    (20, 257, 64, "gemm_strip"), (9, 300, 16390, "gemm_strip"), (65, 333, 700, "gemm_strip"),
    (40, 255, 300, "gemm_mfma"), (40, 700, 63, "gemm_mfma"), (8, 1200, 901, "gemm_mfma"), (33, 1879, 500, "gemm_mfma"), (7, 3992, 531, "gemm_mfma"),  # beside the rule
])
def test_strip_products(hip, oracle, d, m, k, n, path):
    rng = np.random.default_rng(m + k + n)
    a, b = encode(rng.standard_normal((m, k)), d, oracle), encode(rng.standard_normal((k, n)), d, oracle)
    check(hip, oracle, d, pair(a, d, hip, oracle)[0], pair(b, d, hip, oracle)[0], a, b, f"{m}x{k}x{n}")
    if n % 8 or k % 64:  # (aligned rows of a wide matrix have kernels of their own)
        assert hip.last_path() == path, hip.last_path()
    wide = encode(rng.standard_normal((2, m + 1, k + 3)), d, oracle)  # a batch, rows at any element, B shared
    w = hip.shrink(pair(wide, d, hip, oracle)[0], [(0, 2), (1, m + 1), (3, k + 3)])
    v = wide[:, 1:, 3:]
    check(hip, oracle, d, w, pair(b, d, hip, oracle)[0], v, b, f"batch of {m}x{k}x{n}")


@pytest.mark.parametrize("d", HALVES, ids=lambda d: d.name)
def test_special_values_stay_in_their_rows_and_columns(hip, oracle, d):
    """What a tile reads beside its own elements (rows, columns and k past the edge) reaches no result."""
    rng = np.random.default_rng(1)
    m, k, n = 19, 301, 530
    av, bv = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    av[18, 300], av[2, 5], bv[300, 529], bv[0, 64] = np.inf, np.nan, np.nan, -np.inf
    a, b = encode(av, d, oracle), encode(bv, d, oracle)
    got = decode(logical(hip.matmul(pair(a, d, hip, oracle)[0], pair(b, d, hip, oracle)[0])), d, oracle)
    assert hip.last_path() == "gemm_strip"
    bad = np.zeros((m, n), bool)
    bad[[2, 18], :] = bad[:, [64, 529]] = True
    assert np.array_equal(~np.isfinite(got), bad)


@pytest.mark.parametrize("d", HALVES, ids=lambda d: d.name)
@pytest.mark.parametrize("m,n,k", [(8, 512, 512), (48, 768, 512), (150, 576, 512), (200, 520, 512), (20, 520, 3072)])
def test_linear_equals_its_primitives(hip, oracle, d, m, n, k):
    rng = np.random.default_rng(m + n)
    def tensor(*shape):
        return pair(encode(rng.standard_normal(shape), d, oracle), d, hip, oracle)[0]
    x, r = tensor(2, m, k), tensor(2, m, n)
    ws, bs = [tensor(k, n) for _ in range(3)], [tensor(n) for _ in range(3)]
    apart = []
    for w, b in zip(ws, bs):
        p = hip.matmul(x, hip.expand(hip.reshape(w, (1, k, n)), (2, k, n)))
        assert hip.last_path() == "gemm_strip"
        apart.append(hip.binary("add", p, hip.expand(hip.reshape(b, (1, 1, n)), (2, m, n))))
        same_bits(logical(hip.linear(x, w, b)), logical(apart[-1]), "bias")
        assert hip.last_path() == "linear_strip"
        same_bits(logical(hip.linear(x, w, b, r)), logical(hip.binary("add", apart[-1], r)), "bias and residual")
    eager = [logical(t) for t in apart]
    model = Gpt2(Nx(hip), Config())
    with deferred(hip) as win:
        outs = [model.linear(Linear(w, b), x) for w, b in zip(ws, bs)]
        for got, want in zip(outs, eager):
            same_bits(logical(got), want, "a member of a group")
        assert win.delta()["grouped"] == 3 and hip.last_path() == "linear_strip"
