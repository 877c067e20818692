"""GPU parity of the matrix-core products of several and many tokens (matvec_kw at each block shape its dispatch picks,
matmul_tile) at the edges of their tiles: tokens and rows just past and just short of a tile, one 256-value stage and
an odd number of them, strided rows, non-finite values.

Tolerance: as in test_gpu_matvec -- f32 sums of K terms in any order are within 2^-17 S of the exact value (S the sum of
the terms' magnitudes); the exact value here is a 64-bit product with the dequantized rows. The dual epilogue
propagates that through act(g) u, |silu'| <= 1.1."""
import numpy as np
import pytest

import oracle
from tests.test_gpu_matvec import _abs_terms, _run, _seed, _weights, _x

pytestmark = pytest.mark.gpu

CASES = [  # (fmt, x dtype, T, K, N): the block shape (token tiles x 16-row tiles; "tile" for matmul_tile)
    ("q4_k", "f32", 3, 256, 33), ("q5_k", "f32", 16, 768, 17), ("q6_k", "bf16", 31, 512, 47),  # 1 x 1
    ("q4_k", "f32", 17, 256, 2900), ("q8_0", "f32", 16, 512, 4113), ("q3_k", "bf16", 5, 768, 4113),  # 1 x 2
    ("q4_0", "f32", 33, 256, 2900), ("q2_k", "f32", 16, 256, 8209), ("q5_1", "bf16", 48, 512, 2899),  # 1 x 4
    ("q6_k", "f32", 50, 256, 2900), ("f16", "f32", 33, 192, 2895),  # 2 x 2
    ("q4_k", "f32", 130, 256, 2900), ("q5_0", "bf16", 65, 256, 4113), ("q4_1", "f32", 130, 512, 2897),  # 2 x 4
    ("q4_k", "bf16", 50, 512, 8209), ("q8_0", "f32", 300, 256, 2900), ("bf16", "bf16", 130, 320, 4113),  # 4 x 4
    ("q4_k", "f32", 300, 768, 8209), ("q6_k", "f32", 257, 256, 8257), ("q8_0", "bf16", 449, 256, 14336),  # tile
    ("q2_k", "f32", 321, 256, 8193), ("q5_1", "f32", 300, 512, 8209), ("bf16", "f32", 300, 192, 8209),
    ("bf16", "bf16", 331, 64, 4096), ("f16", "bf16", 500, 128, 4113), ("q3_k", "f32", 300, 256, 8209),
    ("q4_k", "f32", 2, 14336, 33), ("bf16", "f32", 2, 14336, 40),  # two tokens past the VALU kernels' LDS
]
DUAL = [
    ("q4_k", "f32", 17, 256, 37), ("q6_k", "f32", 16, 256, 4113), ("q4_1", "bf16", 65, 512, 2900),
    ("q5_k", "f32", 300, 512, 4113), ("q8_0", "bf16", 130, 256, 8257), ("bf16", "bf16", 65, 192, 8209), ("f16", "f32", 5, 320, 40),
]


@pytest.mark.parametrize("fmt,dx,T,K,N", CASES)
def test_products(device, fmt, dx, T, K, N):
    seed = _seed("kw", fmt, dx, T, K, N)
    raw, W = _weights(fmt, N, K, seed, 1)
    x, x32 = _x(dx, T, K, seed)
    y = _run(fmt, dx, "f32", x, [raw], N, K, x_stride=K + 8, y_stride=N + 3).astype(np.float64)
    ref = x32.astype(np.float64) @ W.astype(np.float64).T
    S = np.abs(x32).astype(np.float64) @ _abs_terms(fmt, raw, W).T
    bad = np.abs(y - ref) > 2.0 ** -17 * S + 1e-30
    assert not bad.any(), f"{bad.sum()} of {bad.size} beyond the bound; first at {np.argwhere(bad)[0]}"


@pytest.mark.parametrize("fmt,dx,T,K,N", DUAL)
def test_pairs(device, fmt, dx, T, K, N):
    seed = _seed("kw2", fmt, dx, T, K, N)
    rg, Wg = _weights(fmt, N, K, seed, 1)
    ru, Wu = _weights(fmt, N, K, seed, 2)
    x, x32 = _x(dx, T, K, seed)
    y = _run(fmt, dx, "f32", x, [rg, ru], N, K, act="silu").astype(np.float64)
    xd, ax = x32.astype(np.float64), np.abs(x32).astype(np.float64)
    g, u = xd @ Wg.astype(np.float64).T, xd @ Wu.astype(np.float64).T
    with np.errstate(over="ignore"):
        s = g / (1.0 + np.exp(-g))
    e = 2.0 ** -17
    tol = e * (1.1 * np.abs(u) * (ax @ _abs_terms(fmt, rg, Wg).T) + np.abs(s) * (ax @ _abs_terms(fmt, ru, Wu).T)) + 1e-5 * np.abs(s * u) + 1e-30
    bad = np.abs(y - s * u) > tol
    assert not bad.any(), f"{bad.sum()} of {bad.size} beyond the bound; first at {np.argwhere(bad)[0]}"


@pytest.mark.parametrize("fmt,dx,T,N", [("bf16", "f32", 19, 40), ("f16", "f32", 19, 40), ("f16", "f32", 300, 8209), ("bf16", "bf16", 300, 8209)])
def test_non_finite(device, fmt, dx, T, N):
    """Infinities and NaN come out where the sums have them: in x for both formats, in the weights for f16."""
    K = 128
    raw, W = _weights(fmt, N, K, 5, 1)
    x, x32 = _x(dx, T, K, 5)
    x32 = x32.copy()
    x32[2, 5], x32[4, 70], x32[T - 1, 100] = np.inf, np.nan, -np.inf
    x = x32 if dx == "f32" else oracle.to_bf16(x32)
    if fmt == "f16":
        h = raw.view(np.float16).reshape(N, K).copy()
        h[7, 3], h[N - 1, 90], h[11, 64] = np.inf, -np.inf, np.nan
        raw, W = h.view(np.uint8).reshape(raw.shape), h.astype(np.float32)
    y = _run(fmt, dx, "f32", x, [raw], N, K)
    with np.errstate(invalid="ignore"):
        ref = x32.astype(np.float64) @ W.astype(np.float64).T
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(y[inf].astype(np.float64), ref[inf]) and np.isfinite(y[~inf & ~np.isnan(ref)]).all()
