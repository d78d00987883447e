"""The conduction gather from LDS (uniform smoothing lengths, both precision
modes) and the one from HBM that lengths differing within a material keep.

Tolerance of the run against the oracle: 1e-8 normwise, the FP64 bar of the
thermal tests."""
import numpy as np
import pytest

from oracle_case import normwise_err, oracle_from_case
from weldform_amd import capi, cases

pytestmark = pytest.mark.gpu


def _run(c, steps, **kw):
    s = cases.make_solver(c, **kw)
    s.step(steps)
    s.sync()
    out = {f: s.get(f) for f in ("T", "dTdt", "disp")}
    s.close()
    return out


@pytest.mark.parametrize("precision", [capi.FP64, capi.MIXED])
def test_tiles_from_lds_and_hbm_agree(precision):
    """Every tile from LDS, only those with small sets, or none: the same
    heating bit for bit (4,524 particles, the last tile ragged)."""
    c = cases.thermal_small(steps=20)
    print("n", c.n, "precision", precision, flush=True)
    ref = _run(c, 20, precision=precision, lanes=4)
    for stage in (-1, 300, 600):
        got = _run(c, 20, precision=precision, lanes=4, stage_max=stage)
        for f in ref:
            assert np.array_equal(ref[f], got[f]), (f, stage)


@pytest.mark.parametrize("uniform", [True, False])
def test_heating_matches_oracle(uniform):
    c = cases.thermal_small(steps=20)
    if not uniform:
        c.h = c.h * (1.0 - 0.02 * (np.arange(c.n) % 3))
    print("n", c.n, "uniform h", uniform, flush=True)
    got = _run(c, 20)
    d = oracle_from_case(c, threads=4)
    d.solve_init(c.dt)
    for _ in range(20):
        d.step()
    assert normwise_err(got["T"] - 300.0, d.f("T") - 300.0) < 1e-8
    assert normwise_err(got["disp"], d.f("DISP")) < 1e-8


@pytest.mark.parametrize("precision", [capi.FP64, capi.MIXED])
def test_lone_particle_without_conductivity(precision):
    """A particle with no neighbours takes its heat source alone, whatever
    its material's conductivity: 0 makes the pair factor 0/0, as in the
    reference, but there is no pair."""
    c = cases.thermal_small(steps=2)
    c.thbc = c.hconv = c.tinf = None
    far = c.x.max(axis=0) + 10 * c.meta["dx"]
    for f, v in (("x", far), ("h", c.h[0]), ("mass", c.mass[0]), ("density", c.density[0]), ("ids", 0),
                 ("material", 1), ("sigmay", c.sigmay[0]), ("T", 300.0)):
        setattr(c, f, np.concatenate([getattr(c, f), np.asarray([v], dtype=getattr(c, f).dtype)]))
    c.materials[1] = dict(c.materials[0], k_T=0.0)
    c.dom_max, c.dom_min = (-1e11,) * 3, (1e11,) * 3
    s = cases.make_solver(c, precision=precision)
    q = np.zeros(c.n)
    q[-1] = 1e9
    s.set("q_source", q)
    print("n", c.n, "precision", precision, flush=True)
    s.step(2)
    s.sync()
    assert s.get_int("nb")[-1] == 0
    assert s.get("dTdt")[-1] == pytest.approx(1e9 / (c.density[-1] * c.materials[1]["cp_T"]), rel=1e-12)
    assert np.isfinite(s.get("T")).all()
    s.close()
