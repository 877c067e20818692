"""The float-rows products of several tokens at the limits of their dispatch: rows too long for one token, the switches that
say from how many tokens on the matrix cores are taken, and rows whose bytes or
values pass 32 bits, and activations at the ends of f32."""
import numpy as np
import pytest

from sharplight_amd import native
from tests.devutil import Dev, log
from tests.test_gpu_matvec import _run, _seed, _weights, _x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,T,K,dual", [
    ("q4_k", 2, 24576, False), ("q4_k", 5, 24832, False), ("q8_0", 2, 18944, False), ("q8_0", 17, 19200, False),
    ("q6_k", 3, 20736, False), ("q4_0", 2, 24576, True), ("q2_k", 100, 30720 + 512, True),
])
def test_long_rows_refused(device, fmt, T, K, dual):
    """Rows that the one-token kernels cannot hold: refused at two tokens, and from three for K off the formats' 512 or 1024."""
    N = 16
    with Dev() as d:
        raw, _ = _weights(fmt, N, K, 1, 1)
        px, pw, py = d.empty(T * K * 4), d.put(raw), d.empty(T * N * 4)
        log(f"refusal {fmt} T={T} K={K} dual={dual}")
        with pytest.raises(native.SlhipNotSupported, match="does not fit in LDS"):
            if dual:
                native.dual_matvec("silu", fmt, "f32", "f32", px, T, K, pw, pw, N, py)
            else:
                native.matvec(fmt, "f32", "f32", px, T, K, pw, N, py)


@pytest.mark.parametrize("fmt,T,K", [("q4_k", 3, 24576), ("q8_0", 3, 18944), ("q6_k", 20, 20992)])
def test_long_rows_taken(device, fmt, T, K):
    N = 33
    seed = _seed("long", fmt, T, K)
    raw, W = _weights(fmt, N, K, seed, 1)
    x, x32 = _x("f32", T, K, seed)
    y = _run(fmt, "f32", "f32", x, [raw], N, K).astype(np.float64)
    ref = x32.astype(np.float64) @ W.astype(np.float64).T
    assert np.abs(y - ref).max() <= 2.0 ** -17 * K * np.abs(W).max() * np.abs(x32).max()


@pytest.mark.parametrize("fmt,name,K", [("bf16", "SLHIP_MATVEC_MFMA_MIN_T", 16384), ("f16", "SLHIP_MATVEC_MFMA_MIN_T", 8192),
                                        ("q8_0", "SLHIP_MATVEC_MQ_MIN_T", 14336), ("q4_k", "SLHIP_MATVEC_KQ_MIN_T", 16384)])
@pytest.mark.parametrize("T", [2, 5])
def test_switches_hold_for_long_rows(device, monkeypatch, fmt, name, K, T):
    """Below the switch's token count the VALU kernel runs, also where it holds one token's x at a time: every token's row is
    then the one-token result, bit for bit."""
    monkeypatch.setenv(name, "100")
    monkeypatch.setenv("SLHIP_KQ_MFMA", "0")
    N = 17
    seed = _seed("switch", fmt, T, K)
    raw, _ = _weights(fmt, N, K, seed, 1)
    x, _ = _x("f32", T, K, seed)
    y = _run(fmt, "f32", "f32", x, [raw], N, K)
    for t in range(T):
        assert np.array_equal(y[t].view(np.uint32), _run(fmt, "f32", "f32", x[t:t + 1], [raw], N, K)[0].view(np.uint32)), t


@pytest.mark.parametrize("K,N", [(512 * 526400, 16), (2 ** 31 + 1024, 1)])  # rows of 286 MB (16 of them past 2^32 bytes); values past 2^31
def test_rows_past_32_bits(device, K, N):
    """Q8_0 rows and x of zeros but for a few blocks, at the ends of the first and last row: the sums are those blocks'."""
    T, wrow = 3, K // 32 * 34
    rng = np.random.default_rng(7)
    ref = np.zeros((T, N))
    with Dev() as d:
        log(f"q8_0 K={K} N={N} T={T}: {N * wrow >> 20} MiB of weights, {T * K * 2 >> 20} MiB of x")
        pw, px, py = d.empty(N * wrow, fill=0), d.empty(T * K * 2, fill=0), d.empty(T * N * 4)
        for b in {0, 5, K // 64, K // 32 - 1}:
            xb = rng.integers(-8, 9, (T, 32)).astype(np.float32)
            for t in range(T):
                x16 = np.ascontiguousarray(xb[t].view(np.uint32) >> 16).astype(np.uint16)
                native.call("slhip_memcpy_h2d", px + (t * K + 32 * b) * 2, x16.ctypes.data, 64, None)
                native.synchronize()
            for n in {0, N - 1}:
                q = rng.integers(-127, 128, 32).astype(np.int8)
                block = np.concatenate([np.float16([1.0]).view(np.int8), q])
                native.call("slhip_memcpy_h2d", pw + n * wrow + 34 * b, block.ctypes.data, 34, None)
                native.synchronize()
                ref[:, n] += xb @ q.astype(np.float64)
        native.matvec("q8_0", "bf16", "f32", px, T, K, pw, N, py)
        native.synchronize()
        assert np.array_equal(d.get(py, (T, N), np.float32), ref)


@pytest.mark.parametrize("fmt,T,K,N", [("f16", 3, 256, 40), ("f16", 19, 320, 2900), ("f16", 300, 192, 8209), ("bf16", 2, 8448, 33),
                                       ("bf16", 16, 256, 40), ("bf16", 300, 128, 8209), ("bf16", 5, 512, 20490)])
def test_largest_activations(device, fmt, T, K, N):
    """x of f32's lowest and highest value (as masks have them) times weights small enough: finite sums within f32 rounding,
    on matvec_kw and matmul_tile."""
    big = np.finfo(np.float32).max
    seed = _seed("largest", fmt, T, K, N)
    raw, W = _weights(fmt, N, K, seed, 1)
    x, _ = _x("f32", T, K, seed)
    x = x.copy()
    x[0, 3], x[1, K - 1], x[T - 1, 70], x[T // 2, 40] = -big, big, np.float32(3.397e38), -big
    y = _run(fmt, "f32", "f32", x, [raw], N, K).astype(np.float64)
    ref = x.astype(np.float64) @ W.astype(np.float64).T
    S = np.abs(x).astype(np.float64) @ np.abs(W).astype(np.float64).T
    fits = S < 0.99 * big
    assert fits[[0, 1]].any()
    bad = np.abs(y - ref)[fits] > 2.0 ** -17 * S[fits] + 1e-30
    assert not bad.any() and np.isfinite(y[fits]).all()
    over = np.abs(ref) > 1.01 * big
    assert np.isinf(y[over]).all()
