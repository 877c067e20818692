"""The small copies of a compiled segment (through its pinned staging memory) at their edges: sizes that are no multiple of
16 bytes, runs of other sizes than the compiled one, more inputs than the staging holds at once, inputs set again before
and between runs, and sizes past it, which take the runtime's copies. Every result bit for bit."""
import time

import numpy as np
import pytest

from sharplight_amd import provider, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev(device):
    p = provider.HipExecutionProvider()
    return p.open_device(p.get_devices()[0])


@pytest.mark.parametrize("D,bound", [(1, 5), (3, 7), (1023, 64), (4096, 16), (4099, 33)])
def test_round_trip(dev, D, bound):
    g = provider.GraphBuilder()
    x, z = g.input("f32", "T", D), g.input("f32", "T", D)
    y = g.output(g.add(x, z))
    with dev.compile(g, max_tokens=bound) as seg:
        for k, T in enumerate((bound, 1, bound - 1, bound)):
            a, b = synth.normal(k, 1, (T, D)), synth.normal(k, 2, (T, D))
            seg.set_input(x, synth.normal(9, 9, (T, D)))  # replaced before the run
            seg.set_input(x, a)
            seg.set_input(z, b)
            seg.execute(T)
            assert np.array_equal(seg.get_output(y), a + b)
            seg.set_input(z, a)  # the other input stays
            seg.execute(T)
            seg.set_input(z, b)  # after a run that nothing has waited for
            assert np.array_equal(seg.get_output(y), a + a)


def test_more_inputs_than_the_staging(dev):
    T, D = 16, 1024  # 64 KB each, six of them
    g = provider.GraphBuilder()
    xs = [g.input("f32", "T", D) for _ in range(6)]
    s = xs[0]
    for v in xs[1:]:
        s = g.add(s, v)
    y = g.output(s)
    with dev.compile(g, max_tokens=T) as seg:
        for k in range(3):
            hs = [synth.normal(k, i, (T, D)) for i in range(6)]
            for v, h in zip(xs, hs):
                seg.set_input(v, h)
            seg.execute(T)
            ref = hs[0]
            for h in hs[1:]:
                ref = ref + h
            assert np.array_equal(seg.get_output(y), ref)


def test_a_runs_error_reaches_the_next_call(dev):
    g = provider.GraphBuilder()
    tbl, ids = g.weight("f32", 10, 64), g.input("i32", "T")
    y = g.output(g.gather(tbl, ids))
    with dev.compile(g, max_tokens=4) as seg:
        t = synth.normal(1, 1, (10, 64))
        seg.set_input(tbl, t)
        seg.set_input(ids, np.array([1, 12], np.int32))
        seg.execute(2)
        with pytest.raises(IndexError, match="12"):
            seg.set_input(ids, np.array([1, 2], np.int32))
        seg.set_input(ids, np.array([1, 2], np.int32))
        seg.execute(2)
        assert np.array_equal(seg.get_output(y), t[[1, 2]])


def test_closing_a_segment_keeps_the_error_of_another(dev):
    g = provider.GraphBuilder()
    tbl, ids = g.weight("f32", 10, 64), g.input("i32", "T")
    y = g.output(g.gather(tbl, ids))
    other = dev.compile(g, max_tokens=4)
    with dev.compile(g, max_tokens=4) as seg:
        seg.set_input(tbl, synth.normal(1, 1, (10, 64)))
        seg.set_input(ids, np.array([1, 12], np.int32))
        seg.execute(2)
        time.sleep(0.2)  # the run has ended, nothing has waited for it
        other.close()
        with pytest.raises(IndexError, match="12"):
            seg.get_output(y)
