"""Adaptive time stepping on the GPU against the CPU oracle: CheckMinTSVel
(smallest neighbour distance, CFL d / (Cs + |v|)), CheckMinTSAccel
(sqrt_h_a sqrt(h / |a|), the later check, so it wins when both are on) and
AdaptiveTimeStep's harmonic blend (Source/Domain.cpp:206-319), evaluated
between the two halves of the kick (Source/SolverLeapfrog.cpp:256-262,
Source/SolverKickDrift.cpp:214-226).  The step size lives on the device, so
the amplitude-driven BC also checks that the device clock advances by the
adapted steps.

Bars: FP64 step sizes within 1e-10 relative at every step, displacement and
reaction history within 1e-8 normwise; mixed precision step sizes within
1e-4 relative, displacement within 1e-4."""
import numpy as np
import pytest

from oracle_case import normwise_err, oracle_from_case
from weldform_amd import capi, cases

pytestmark = pytest.mark.gpu

STEPS = 100


def _case(auto_ts):
    # initial dt = h / Cs, above the velocity limit 0.7 dx / Cs, so the
    # velocity criterion cuts it at once; the acceleration criterion (with the
    # reference's sqrt_h_a = 0.0025) cuts it further once the ramp moves the top
    c = cases.cylinder_case("cyl_upset_4k_jc_auto_ts", 7.5e-3, 30e-3, 1.0e-3, cases.AL["rho"], cases.AL["E"],
                            cases.AL["nu"], cases.JC_AL, dt_cfl=1.0, steps=STEPS, jitter=1e-3, seed=7,
                            v_top=-20.0, T0=300.0)
    c.amps = [dict(id=1, t=[0.0, 40 * c.dt, 1.0], v=[0.0, 1.0, 1.0])]
    c.bcs[1].update(value_type=1, amp_id=1, amp_factor=1.0)
    c.auto_ts = auto_ts
    return c


_ORACLE = {}


def _oracle(auto_ts, scheme):
    key = (auto_ts, scheme)
    if key not in _ORACLE:
        c = _case(auto_ts)
        d = oracle_from_case(c, threads=8)
        d.solve_init(c.dt)
        dts, R = [], []
        for _ in range(c.steps):
            d.step(scheme)
            dts.append(d.param("deltat"))
            R.append(d.reaction(c.top_zone).copy())
        _ORACLE[key] = (c, d, np.array(dts), np.array(R))
    return _ORACLE[key]


@pytest.mark.parametrize("auto_ts,scheme,precision", [
    (1, "leapfrog", capi.FP64), (3, "leapfrog", capi.FP64), (1, "kickdrift", capi.FP64),
    (1, "leapfrog", capi.MIXED), (3, "leapfrog", capi.MIXED)])
def test_adaptive_step_matches_oracle(auto_ts, scheme, precision):
    c, d, dts, R = _oracle(auto_ts, scheme)
    print(f"adaptive dt: n={c.n} steps={c.steps} auto_ts={auto_ts} scheme={scheme} precision={precision}",
          flush=True)
    assert dts.min() < 0.7 * c.dt  # the step did adapt
    g = cases.make_solver(c, precision=precision)
    sch = capi.LEAPFROG if scheme == "leapfrog" else capi.KICKDRIFT
    got = []
    for _ in range(c.steps):
        g.step(1, sch)
        got.append(g.scalars()["dt"])
    g.sync()
    got = np.array(got)
    sc = g.scalars()
    fp64 = precision == capi.FP64
    dt_err = np.abs(got / dts - 1).max()
    errs = {"disp": normwise_err(g.get("disp"), d.f("DISP")),
            "reaction": normwise_err(g.reaction_history(c.top_zone)[:, 2], R[:, 2])}
    print("dt rel err", dt_err, "time", sc["time"], d.param("Time"), errs, flush=True)
    assert dt_err < (1e-10 if fp64 else 1e-4)
    assert sc["time"] == pytest.approx(d.param("Time"), rel=1e-10 if fp64 else 1e-4)
    assert errs["disp"] < (1e-8 if fp64 else 1e-4)
    if fp64:
        assert errs["reaction"] < 1e-8


# Models of more than 320 tiles (40,960 particles) update the stress in a kernel
# of its own, smaller ones at the end of the rate kernel: a billet a little
# larger, whose soft metal flows from the first step, against the oracle.
# Bars: rounding over a few steps, FP64 as above; the temperature's change is
# 1e-6 of the temperature, so its bar is 1e-6; in mixed precision the FP32
# records put 1e-5 on the strain rates, 1e-3 bounds the stress and the heat made of them.
LARGE_STEPS = 6
SOFT = dict(cases.JC_AL, jc_A=2e6, jc_B=20e6, k_T=130.0, cp_T=900.0, th_exp=2.3e-5)


def _large_case(opt):
    c = cases.cylinder_case("cyl_flow_auto_ts", 7.5e-3, 30e-3, 0.47e-3, cases.AL["rho"], cases.AL["E"],
                            cases.AL["nu"], SOFT, dt_cfl=1.0, steps=LARGE_STEPS, jitter=1e-3, seed=7,
                            v_top=-60.0, T0=300.0)
    z, rate = c.x[:, 2], 60.0 / 30e-3
    c.v = np.stack([0.5 * rate * c.x[:, 0], 0.5 * rate * c.x[:, 1], -rate * (z - z.min())], axis=1)
    c.auto_ts = 1
    if opt == "thermal":
        c.thermal = c.pl_heating = True
    if opt == "damage":
        c.damage = {0: (0.02, 0.03, -2.0, 0.01, 0.4)}
    return c


_LARGE = {}


def _large_oracle(opt, scheme):
    if (opt, scheme) not in _LARGE:
        c = _large_case(opt)
        d = oracle_from_case(c, threads=8)
        d.solve_init(c.dt)
        dts = []
        for _ in range(c.steps):
            d.step(scheme)
            dts.append(d.param("deltat"))
        _LARGE[opt, scheme] = (c, d, np.array(dts))
    return _LARGE[opt, scheme]


@pytest.mark.parametrize("opt,scheme,precision", [
    ("", "leapfrog", capi.FP64), ("", "kickdrift", capi.FP64), ("", "leapfrog", capi.MIXED),
    ("", "kickdrift", capi.MIXED), ("thermal", "leapfrog", capi.FP64), ("thermal", "leapfrog", capi.MIXED),
    ("damage", "leapfrog", capi.FP64)])
def test_adaptive_step_with_a_separate_stress_update(opt, scheme, precision):
    c, d, dts = _large_oracle(opt, scheme)
    print(f"adaptive dt, large: n={c.n} steps={c.steps} {opt} scheme={scheme} precision={precision}", flush=True)
    assert c.n > 320 * 128 and dts.max() < 0.8 * c.dt
    assert np.median(d.f("PLSTRAIN")) > 1e-5
    g = cases.make_solver(c, precision=precision)
    g.step(c.steps, capi.LEAPFROG if scheme == "leapfrog" else capi.KICKDRIFT)
    g.sync()
    fp64 = precision == capi.FP64
    tol = 1e-8 if fp64 else 1e-4
    want = [("strain", "STRAIN", tol), ("pl_strain", "PLSTRAIN", tol), ("disp", "DISP", tol),
            ("sigma", "SIGMA", tol if fp64 else 1e-3)]
    if opt == "damage":
        want.append(("dam_D", "DAMD", tol))
    got = {f: (normwise_err(g.get(f).reshape(-1), d.f(o).reshape(-1)), t) for f, o, t in want}
    if opt == "thermal":
        got["T"] = (normwise_err(g.get("T") - 300.0, d.f("T") - 300.0), 1e-6 if fp64 else 1e-3)
    got["time"] = (abs(g.scalars()["time"] / d.param("Time") - 1), 1e-10 if fp64 else 1e-4)
    print(got, flush=True)
    for f, (e, t) in got.items():
        assert e < t, f
