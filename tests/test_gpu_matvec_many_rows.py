"""GPU parity of the several-token products whose dispatch begins at many rows: the LDS-staged kernel of bf16 weights
(matvec_mfma_lds) just past the row counts from which it is taken, and matvec_mq2 of the block formats, with ragged row
tiles, every format, both activation types, single matrices and pairs. And what a token with non-finite
activations does to the others, on these kernels, matvec_kw and matmul_tile.

Tolerance: as in test_gpu_matvec_kw."""
import numpy as np
import pytest

import oracle
from tests.test_gpu_matvec import _run, _seed, _weights, _x
from tests.test_gpu_matvec_kw import test_pairs as check_pair, test_products as check_product

pytestmark = pytest.mark.gpu

MQ = ["q4_0", "q8_0", "q4_1", "q5_0", "q5_1", "q4_k", "q5_k", "q6_k", "q2_k", "q3_k"]


@pytest.mark.parametrize("dx,T,K,N", [("bf16", 2, 256, 16391), ("bf16", 16, 512, 16391), ("bf16", 9, 768, 16385), ("bf16", 8, 2304, 6151)])
def test_bf16_rows(device, dx, T, K, N):
    check_product(device, "bf16", dx, T, K, N)


@pytest.mark.parametrize("dx,T,K,N", [("bf16", 2, 512, 4105), ("bf16", 16, 256, 4105), ("f32", 3, 512, 8201), ("f32", 13, 256, 8201),
                                      ("f32", 16, 768, 8193)])  # f32 x: one row tile a block up to 12 tokens, two above
def test_bf16_pairs(device, dx, T, K, N):
    check_pair(device, "bf16", dx, T, K, N)


@pytest.mark.parametrize("stage,tiles", [("512", "1"), ("256", "1"), ("256", "2")])
@pytest.mark.parametrize("dx,N", [("f32", 8201), ("bf16", 4105)])
def test_bf16_stages(device, monkeypatch, stage, tiles, dx, N):
    """Each stage width and tile count that the switches select."""
    monkeypatch.setenv("SLHIP_MATVEC_MFMA_SK", stage)
    monkeypatch.setenv("SLHIP_MATVEC_MFMA_NT", tiles)
    check_pair(device, "bf16", dx, 11, 1024, N)


@pytest.mark.parametrize("fmt", MQ)
@pytest.mark.parametrize("dx,T", [("f32", 3), ("f32", 16), ("bf16", 16)])
def test_block_format_rows(device, fmt, dx, T):
    check_product(device, fmt, dx, T, 1024, 16391)


@pytest.mark.parametrize("fmt", MQ)
@pytest.mark.parametrize("dx,T", [("f32", 16), ("bf16", 3)])
def test_block_format_pairs(device, fmt, dx, T):
    check_pair(device, fmt, dx, T, 1024, 8201)


@pytest.mark.parametrize("fmt,dx,T,K,N,pair", [
    ("q6_k", "f32", 7, 1536, 8203, False), ("q2_k", "f32", 16, 3072, 8201, True), ("q3_k", "f32", 3, 512, 8201, True),  # the narrower stages
    ("q8_0", "bf16", 5, 512, 8203, True), ("q6_k", "bf16", 16, 512, 16385, False), ("q8_0", "f32", 17, 512, 8201, True), ("q4_1", "bf16", 32, 1024, 8201, True),  # two launches
])
def test_few_stages(device, fmt, dx, T, K, N, pair):
    (check_pair if pair else check_product)(device, fmt, dx, T, K, N)


@pytest.mark.parametrize("fmt,dx,T,K,N", [
    ("q4_k", "f32", 19, 256, 40), ("q6_k", "f32", 19, 512, 40), ("q8_0", "bf16", 19, 512, 40), ("q2_k", "f32", 33, 256, 2900),  # matvec_kw
    ("q3_k", "f32", 19, 256, 40), ("q5_1", "f32", 50, 256, 2900),
    ("q4_k", "f32", 300, 256, 8209), ("q6_k", "f32", 257, 256, 8257), ("q2_k", "f32", 321, 256, 8193), ("q8_0", "bf16", 449, 256, 14336),  # tile
    ("q4_0", "f32", 16, 1024, 16391), ("q5_1", "bf16", 16, 1024, 16391), ("bf16", "bf16", 16, 256, 16391),  # mq2, LDS-staged
    ("q6_k", "bf16", 16, 1024, 8209), ("q5_k", "f32", 8, 1024, 16391), ("q2_k", "bf16", 9, 1024, 8209),
])
def test_a_non_finite_token_leaves_the_others(device, fmt, dx, T, K, N):
    """A token with an infinity or NaN among its activations comes out non-finite in every row, and all other tokens' rows
    are bit for bit what they are without it."""
    seed = _seed("non-finite", fmt, dx, T, K, N)
    raw, _ = _weights(fmt, N, K, seed, 1)
    _, x = _x(dx, T, K, seed)
    x = x.copy()
    put = (lambda v: v) if dx == "f32" else oracle.to_bf16
    clean = _run(fmt, dx, "f32", put(x), [raw], N, K)
    bad = [1, 6, T - 1]
    x[1, 5], x[6, K - 9], x[T - 1, 40] = np.inf, np.nan, -np.inf
    y = _run(fmt, dx, "f32", put(x), [raw], N, K)
    assert not np.isfinite(y[bad]).any()
    rest = np.setdiff1d(np.arange(T), bad)
    assert np.array_equal(y[rest].view(np.uint32), clean[rest].view(np.uint32)) and np.isfinite(clean).all()
