"""The float-rows products of several tokens at the limits of their dispatch: rows too long for one token, the switches that
say from how many tokens on the matrix cores are taken."""
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
