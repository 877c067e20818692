"""GPU parity of the several-token integer-dot product (matvec_kw8) at the edges of its tiles and of its dispatch: tokens
and rows just past and just short of a tile, fewer 256-value stages than waves and an odd number of them, both block
sizes, and the sizes just past the dispatch's lines, which the row-resident kernels keep.

Tolerance: as in test_gpu_matvec_q8 -- 2^-16 S of the oracle, S the sum of the terms' magnitudes per 16 values; the dual
epilogue propagates that through act(g) u, |silu'| <= 1.1."""
import numpy as np
import pytest

import oracle
from sharplight_amd import native, synth
from tests.devutil import Dev
from tests.test_gpu_matvec_q8 import _act64, _compare, _run, _seed, _x

pytestmark = pytest.mark.gpu

FORMATS = ["q4_0", "q4_1", "q5_0", "q5_1", "q8_0", "iq4_nl", "q4_k", "q5_k", "q6_k"]
SINGLE = [
    *[(f, "f32", 5, 256, 17) for f in FORMATS],      # one stage: seven waves idle
    *[(f, "bf16", 31, 2304, 47) for f in FORMATS],   # nine stages, two token tiles, a short row tile
    *[(f, "f32", 17, 512, 8209) for f in FORMATS],   # many row tiles (two to a block where the format takes them)
    *[(f, "f32", 5, 512, 16401) for f in FORMATS],   # past the line for few tokens
    ("q4_k", "f32", 3, 14336, 33), ("q4_0", "f32", 3, 768, 1), ("q6_k", "f32", 4, 8192, 40), ("q8_0", "f32", 3, 8192, 40),
    ("iq4_nl", "bf16", 16, 256, 16401), ("q4_k", "f32", 100, 256, 8193), ("q5_1", "f32", 17, 256, 32785), ("q6_k", "f32", 5, 768, 16401),
]
SINGLE += [*[(f, "f32", 17, 2048, 8209) for f in FORMATS]]  # many row tiles, an even split of the stages
PAIRS = [
    *[(f, 16, 512, 33) for f in FORMATS],
    *[(f, 17, 256, 8209) for f in FORMATS],
    ("q4_k", 5, 256, 8209), ("q8_0", 16, 256, 4113), ("q6_k", 31, 2304, 16),
    *[(f, 17, 2048, 4113) for f in FORMATS], ("q4_0", 9, 2048, 16401), ("iq4_nl", 9, 2048, 8209), ("q4_k", 9, 2048, 8209),
]


@pytest.mark.parametrize("fmt,dx,T,K,N", SINGLE)
def test_products(device, fmt, dx, T, K, N):
    seed = _seed("kw8", fmt, dx, T, K, N)
    raw = synth.quant_table(fmt, N, K, seed=seed, tid=1)
    x, x32 = _x(dx, T, K, seed, spread=dx == "f32")
    b = synth.normal(seed, 4, (N,), dtype="f32")
    y = _run(fmt, dx, "f32", x, [raw], N, K, bias=b)
    ref, S = oracle.matvec_q8(fmt, raw, N, K, x32, with_abs=True)
    ref = oracle.add(ref, np.broadcast_to(b, ref.shape).copy())
    _compare(y, "f32", ref, 2.0 ** -16 * S + 2.0 ** -24 * np.abs(ref) + 1e-30, f"matvec_q8 {fmt}")


@pytest.mark.parametrize("fmt,T,K,N", PAIRS)
def test_pairs(device, fmt, T, K, N):
    seed = _seed("kw8 pair", fmt, T, K, N)
    raws = [synth.quant_table(fmt, N, K, seed=seed, tid=t) for t in (1, 2)]
    x, x32 = _x("f32", T, K, seed)
    y = _run(fmt, "f32", "bf16", x, raws, N, K, act="silu")
    (g, Sg), (u, Su) = (oracle.matvec_q8(fmt, r, N, K, x32, with_abs=True) for r in raws)
    ref = oracle.mul(oracle.unary("silu", g), u)
    tol = 2.0 ** -16 * (1.1 * np.abs(u) * Sg + np.abs(_act64("silu", g)) * Su) + 1e-5 * np.abs(ref) + 1e-30
    _compare(y, "bf16", ref, tol, f"dual_matvec_q8 {fmt}")


def test_refusals_stand(device):
    """Rows too long for the one-token kernel's LDS are refused for several tokens as for one."""
    K, N = 256 * 641, 16
    with Dev() as d:
        px, pw, py = d.empty(8 * native.q8_row_bytes(K)), d.empty(N * K // 256 * 210), d.empty(8 * N * 4)
        for T in (1, 8):
            with pytest.raises(native.SlhipNotSupported, match="does not fit in LDS"):
                native.matvec_q8("q6_k", "f32", px, T, K, pw, N, py)
