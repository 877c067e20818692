"""GPU parity of the integer-dot matvec where two waves share a long row (one and two tokens): one row, odd row counts that
leave a wave pair idle in the last round, several rounds, and pairs. Tolerance as in test_gpu_matvec_q8."""
import numpy as np
import pytest

import oracle
from sharplight_amd import synth
from tests.test_gpu_matvec_q8 import _act64, _compare, _run, _seed, _x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,T,K,N", [
    ("q4_k", 1, 14336, 1), ("q4_k", 1, 14336, 4099), ("q4_k", 2, 16384, 5), ("q5_k", 2, 14336, 2051), ("q8_0", 1, 14336, 7),
    ("q8_0", 2, 8192, 2051), ("q5_1", 2, 14336, 33), ("q4_0", 1, 16384, 3), ("iq4_nl", 1, 14336, 34), ("mxfp4", 2, 16384, 35),
    ("q6_k", 1, 16384, 2049), ("q4_1", 1, 14336, 1025),
])
def test_shared_rows(device, fmt, T, K, N):
    seed = _seed("parts", fmt, T, K, N)
    raw = synth.quant_table(fmt, N, K, seed=seed, tid=1)
    x, x32 = _x("f32", T, K, seed)
    b = synth.normal(seed, 4, (N,), dtype="f32")
    y = _run(fmt, "f32", "f32", x, [raw], N, K, bias=b)
    ref, S = oracle.matvec_q8(fmt, raw, N, K, x32, with_abs=True)
    ref = oracle.add(ref, np.broadcast_to(b, ref.shape).copy())
    _compare(y, "f32", ref, 2.0 ** -16 * S + 2.0 ** -24 * np.abs(ref) + 1e-30, f"matvec_q8 {fmt}")


@pytest.mark.parametrize("fmt,T,K,N", [("q8_0", 1, 8192, 2051), ("q8_0", 2, 8192, 3), ("q5_k", 1, 14336, 1)])
def test_shared_pairs(device, fmt, T, K, N):
    seed = _seed("parts pair", fmt, T, K, N)
    raws = [synth.quant_table(fmt, N, K, seed=seed, tid=t) for t in (1, 2)]
    x, x32 = _x("f32", T, K, seed)
    y = _run(fmt, "f32", "f32", x, raws, N, K, act="silu")
    (g, Sg), (u, Su) = (oracle.matvec_q8(fmt, r, N, K, x32, with_abs=True) for r in raws)
    ref = oracle.mul(oracle.unary("silu", g), u)
    tol = 2.0 ** -16 * (1.1 * np.abs(u) * Sg + np.abs(_act64("silu", g)) * Su) + 1e-5 * np.abs(ref) + 1e-30
    _compare(y, "f32", ref, tol, f"dual_matvec_q8 {fmt}")
