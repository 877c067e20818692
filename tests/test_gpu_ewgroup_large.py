"""Row-form groups whose launch is large enough for the streaming loads: every row bit for bit what smaller launches of the
same rows (plain loads) give, for tails and heads, f32 and 16-bit rows, and a row count just past the line."""
import numpy as np
import pytest

from sharplight_amd import native, synth
from tests.devutil import Dev, log

pytestmark = pytest.mark.gpu

NP = {"f32": np.float32, "bf16": np.uint16, "f16": np.float16}
LINE = 144 << 20


def _run(dt, x, r, w, cols, form):
    rows = x.shape[0]
    with Dev() as d:
        log(f"ew group {form} {dt} rows={rows} cols={cols}")
        px, pr, pw = d.put(x), d.put(r), d.put(w)
        n = max(rows * cols * x.dtype.itemsize, 4)
        ph, py = d.empty(n), d.empty(n)
        ins = [(px, dt, native.EWI_FULL), (pr, dt, native.EWI_FULL)]
        op = [("binary", "Add", 0, 1, 2, dt, 0, 0)]
        if form == "tail":
            native.ew_program(ins, op, [(ph, dt, 2)], rows, cols, tail={"kind": "rms", "reg": 2, "w": pw, "eps": 1e-5, "y": py, "dtype_y": dt})
        else:
            native.ew_program(ins, op, [(ph, dt, 2)], rows, cols, head={"kind": "rms", "reg": 0, "w": pw, "eps": 1e-5, "dtype_y": dt})
        native.synchronize()
        out = [d.get(ph, (rows, cols), x.dtype)]
        if form == "tail":
            out.append(d.get(py, (rows, cols), x.dtype))
        return out


@pytest.mark.parametrize("form,dt,cols", [("tail", "f32", 4096), ("tail", "bf16", 1000), ("head", "f32", 260), ("head", "f16", 4096)])
def test_large_equals_small(device, form, dt, cols):
    size = np.dtype(NP[dt]).itemsize
    rows = LINE // ((4 if form == "tail" else 3) * size * cols) + 1
    base = synth.normal(3, 1, (64, cols), dtype=dt).astype(NP[dt], copy=False).reshape(64, cols)
    x = np.tile(base, (rows // 64 + 1, 1))[:rows]
    r = np.roll(x, 7, axis=0)
    w = synth.normal(3, 2, (cols,), 1.0, 0.1)
    whole = _run(dt, x, r, w, cols, form)
    for a in range(0, rows, rows // 3):
        b = min(rows, a + rows // 3)
        for big, small in zip(whole, _run(dt, x[a:b], r[a:b], w, cols, form)):
            assert np.array_equal(big[a:b].view(np.uint8), small.view(np.uint8))
