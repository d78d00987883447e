"""The FP64 pair passes that read each tile's neighbours from LDS, against the
HBM gathers of two lanes (which the parity tests hold to the oracle).

Tolerance: each sum has at most 128 terms of random sign and size, so the two
summation orders and reciprocals differ by a few roundings of the largest
term: 1e-12 normwise."""
import numpy as np
import pytest

from oracle_case import normwise_err
from weldform_amd import capi, cases

pytestmark = pytest.mark.gpu

PASSES = (("accel", ("a",)), ("density", ("ddensity",)), ("rates", ("strain_rate", "rot_rate")))


def _case(n, beta=0.0):
    """The first n particles (whole rows and layers, the last one ragged) of
    a jittered billet of 7 rows' radius."""
    c = cases.small_jc(dx=1.0e-3, seed=n)
    order = np.lexsort((c.x[:, 0], c.x[:, 1], c.x[:, 2]))[:n]
    for f in ("x", "h", "mass", "density", "ids", "material", "sigmay", "T"):
        setattr(c, f, getattr(c, f)[order])
    c.materials[0]["beta"] = beta
    c.dom_max, c.dom_min = (0.02,) * 3, (-0.02,) * 3  # (a single layer has no height of its own)
    return c


def _passes(c, state, **kw):
    s = cases.make_solver(c, **kw)
    s.set("v", state["v"])
    s.set("density", state["rho"])
    s.set("sigma", state["sig"])
    if "D" in state:
        s.set("dam_D", state["D"])
    s.rebuild_neighbours()
    out = {}
    for name, fields in PASSES:
        print("eval", name, "n", c.n, kw, flush=True)
        s.eval(name)
        for f in fields:
            out[f] = s.get(f)
    s.close()
    return out


def _state(c, damage=False):
    rng = np.random.default_rng(c.n)
    s = rng.normal(0.0, 1e8, size=(c.n, 3, 3))
    st = dict(v=rng.normal(0.0, 1.0, size=(c.n, 3)), rho=c.density * (1.0 + 1e-3 * rng.uniform(-1, 1, c.n)),
              sig=0.5 * (s + np.transpose(s, (0, 2, 1))))
    if damage:
        st["D"] = rng.uniform(0.0, 1.3, c.n).clip(0.0, 1.0)
    return st


def _check(a, b):
    for f in a:
        assert normwise_err(a[f], b[f]) < 1e-12, f


@pytest.mark.parametrize("n", [127, 128, 129, 500, 1021, 2049])
def test_tiles(n):
    c = _case(n)
    st = _state(c)
    ref = _passes(c, st, lanes=2)
    got = _passes(c, st)
    _check(got, ref)
    # every tile from LDS, none, or only those with small sets
    for stage in (-1, 300, 600):
        other = _passes(c, st, stage_max=stage)
        for f in got:
            assert np.array_equal(got[f], other[f]), (f, stage)
    same = _passes(c, st, lanes=4)
    for f in got:
        assert np.array_equal(got[f], same[f]), f


@pytest.mark.parametrize("opt", ["beta", "grad_corr", "locking", "damage", "damage_beta", "plate"])
def test_options(opt):
    if opt == "plate":
        c = cases.plate2d_small(steps=1)
    else:
        c = _case(1021, beta=2.0 if "beta" in opt else 0.0)
    if "damage" in opt:
        c.damage = {0: (0.2, 0.3, -2.0, 0.01, 0.4)}
    st = _state(c, "damage" in opt)
    if opt == "plate":
        st["v"][:, 2] = 0.0
    kw = dict(grad_corr=True, locking=True) if opt == "grad_corr" else dict(locking=True) if opt == "locking" else {}
    _check(_passes(c, st, **kw), _passes(c, st, lanes=2, **kw))


def test_lengths_that_differ_gather_from_hbm():
    """Smoothing lengths that differ within a material take the HBM gathers,
    also when they are set after the context was made; uniform ones again
    the passes from LDS."""
    c = _case(500)
    st = _state(c)
    h = c.h * (1.0 - 0.05 * (np.arange(c.n) % 2))
    c.h = h
    ref = _passes(c, st, lanes=2)
    got = _passes(c, st)
    for f in ref:
        assert np.array_equal(ref[f], got[f]), f
    c2 = _case(500)
    uni = _passes(c2, st)
    s = cases.make_solver(c2)
    for hh, want in ((h, ref), (c2.h, uni)):
        s.set("h", hh)
        for f, v in (("v", st["v"]), ("density", st["rho"]), ("sigma", st["sig"])):
            s.set(f, v)
        s.rebuild_neighbours()
        for name, fields in PASSES:
            s.eval(name)
            for f in fields:
                assert np.array_equal(s.get(f), want[f]), (f, name)
    s.close()


def test_lengths_made_uniform_after_init():
    """A context made with lengths that differ and then given uniform ones:
    the passes of a context uniform from the start, bit for bit."""
    c = _case(500)
    st, h = _state(c), c.h
    want = _passes(c, st)
    c.h = h * (1.0 - 0.05 * (np.arange(c.n) % 2))
    s = cases.make_solver(c)
    s.set("h", h)
    for f, v in (("v", st["v"]), ("density", st["rho"]), ("sigma", st["sig"])):
        s.set(f, v)
    s.rebuild_neighbours()
    for name, fields in PASSES:
        s.eval(name)
        for f in fields:
            assert np.array_equal(s.get(f), want[f]), (f, name)
    s.close()


@pytest.mark.parametrize("opt", ["", "thermal", "plate"])
def test_run_does_not_depend_on_staging(opt):
    """Steps with every tile from LDS, none, or those with small sets: the
    state and the scalars, the energies of the rate pass among them, are the
    same bit for bit."""
    ref = None
    for stage in (0, -1, 600):
        c = {"": cases.small_jc, "thermal": cases.thermal_small, "plate": cases.plate2d_small}[opt](steps=12)
        s = cases.make_solver(c, stage_max=stage)
        s.set("pl_strain", np.full(c.n, 0.05))
        print("run", opt, "n", c.n, "stage", stage, flush=True)
        s.step(12)
        s.sync()
        got = {f: s.get(f) for f in ("x", "v", "a", "density", "sigma", "strain", "T", "dTdt")}
        got["scalars"] = sorted(s.scalars().items())
        s.close()
        ref = ref or got
        for f in got:
            assert np.array_equal(got[f], ref[f]), (f, stage)
