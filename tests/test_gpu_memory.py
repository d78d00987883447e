"""FP64 contexts on a device whose memory is short: the staging lists of the
passes from LDS, and the gradient tape's copies of them, are done without, or
given back, where something that a context cannot do without asks for their
memory.  The passes then read the same records from HBM, or lists formed
again, so that the results are the same bit for bit."""
import ctypes
import math

import numpy as np
import pytest

from weldform_amd import capi, cases

pytestmark = pytest.mark.gpu


def _free():
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert capi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


class _Fill:
    """Holds the device's memory down to `leave` bytes."""

    def __init__(self, leave):
        self.held = []
        while True:
            spare = _free() - leave
            if spare < 4 << 20:
                break
            p = ctypes.c_void_p()
            if capi.lib().hipMalloc(ctypes.byref(p), ctypes.c_size_t(min(spare, 16 << 30))) != 0:
                break
            self.held.append(p)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.held:
            assert capi.lib().hipFree(p) == 0


def _case(n=480e3):
    R, L = 15e-3, 30e-3
    return cases.config5_zone(steps=4, dx=(math.pi * R * R * L / n) ** (1 / 3), R=R, L=L, v_top=-5.0, seed=3)


def _solver(c, **kw):
    g = cases.make_solver(c, **kw)
    g.step(2)
    g.sync()
    return g


def _gradient(g):
    loss, hist = g.adj_forward(np.full(4, 1e4), checkpoint_every=2, kind=capi.ADJ_ZONE, index=3, component=2)
    return [np.array([loss]), hist, g.adj_backward(), g.adj_field("x")]


def test_lists_are_given_back():
    g = _solver(_case(4e3))  # (what the runtime itself takes is taken)
    g.pack_xdmf()
    _gradient(g)
    g.close()
    c = _case()
    want, used = {}, {}
    for stage_max in (-1, 0):  # without and with lists, all the memory there
        before = _free()
        g = _solver(c, stage_max=stage_max)
        used["context", stage_max] = before - _free()
        want = dict(state=[g.get("x"), g.get("sigma")], table=g.pack_xdmf())
        before = _free()
        want["gradient"] = _gradient(g)
        used["window", stage_max] = before - _free()
        g.close()
    need, lists = used["context", -1], used["context", 0] - used["context", -1]
    window, half = used["window", -1], lists // 2
    table = 4 * (capi.XDMF_NF + capi.XDMF_NI) * c.n
    print("n", c.n, "MiB: lists", lists >> 20, "window", window >> 20, "table", table >> 20, flush=True)
    assert lists > 128 << 20 and table > 64 << 20
    assert abs(used["window", 0] - window - 2 * lists) < half  # two tape slots' lists
    cases_ = (  # what the device's memory holds, beside the context, and what is asked of it
        ("no lists", need + half, ()),
        ("lists or table", need + lists + table // 2, ("table",)),
        ("lists or window", need + lists + table + window - half, ("table", "gradient")),
        ("lists and window", need + lists + table + window + half, ("table", "gradient")),
        ("the tape's lists or table", need + 3 * lists + window + table // 2, ("gradient", "table", "gradient")))
    with _Fill(8 << 30):
        for what, leave, asked in cases_:
            with _Fill(leave):
                print("case", what, "MiB left", _free() >> 20, flush=True)
                g = _solver(c)
                got = [("state", [g.get("x"), g.get("sigma")])]
                for a in asked:
                    if a == "table":
                        got.append((a, g.pack_xdmf()))
                    else:
                        got.append((a, _gradient(g)))
                        g.adj_restore()
                g.step(2)
                g.sync()
                g.close()
            for name, arrays in got:
                for k, (a, b) in enumerate(zip(arrays, want[name])):
                    assert np.array_equal(a, b), (what, name, k)
