"""Performance cases: stretches of explicit steps as a user's program runs them.

A pass advances a prepared solver by `steps` steps, waits for it and fetches the
output table of the reference's writers (Domain::WriteXDMF, float32), as a
program does at each output of a run; the state of every particle in it
(positions, velocities, densities, stresses, strains, plastic strain,
temperature, ids, neighbour counts) is the pass's result.  The table's rates of
the last step (acceleration, strain rate) are left out: their integrals are
there, and after a smooth flow they are small differences of large sums.  A
pass of an adjoint case runs one window forward and backward and fetches the
gradients.  The state goes on from pass to pass as a simulation does; an
adjoint pass restores the window's start.

The ranges: billets of 1.5 thousand to a million particles, both precisions,
both schemes, fixed and adaptive steps, 3D and plane strain; before yield (one
neighbour search per run) and on worked, yielding stock (a search every five
steps); rigid contact with conduction and plastic heat, damage, a batch of
specimens in one context, and the reverse-mode gradient.
"""
import math

import numpy as np
import torch

from weldform_amd import capi, cases, output

AL = cases.AL


def listed():
    c = []

    def add(name, kind, n, steps, **kw):
        c.append(dict(_default(kind), name=name, n=n, steps=steps, **kw))

    # one small specimen of a calibration, between its punches, already work-hardened: launch latency decides
    add("specimen_2k_mixed", "contact", 1700, 200, precision="mixed", yielding=True, thermal=False)
    # plane strain: the smallest models (a 30 mm x 60 mm plate at 1 mm pitch), parity precision
    add("plate2d_1.9k_fp64", "plate2d", 1891, 200, precision="fp64", yielding=True)
    # the scene driver's and the smoke test's size: an elastic upsetting in FP64
    add("upset_4.5k_fp64", "billet", 4500, 200, precision="fp64", yielding=False)
    # a calibration gradient at test size
    add("adjoint_4.5k", "adjoint", 4500, 60)
    # mid-size scene with the adaptive step and KickDrift, yielding
    add("adaptive_37k_mixed", "billet", 37000, 100, precision="mixed", yielding=True, scheme="kickdrift", adaptive=True)
    # Johnson-Cook damage (FP64, Locking sums, free surface every step)
    add("damage_61k_fp64", "damage", 61000, 60, precision="fp64", yielding=True)
    # the calibration gradient at its full size: window and reverse sweep
    add("adjoint_200k", "adjoint", 200000, 20)
    # forging step: rigid punches, friction, conduction and plastic heat, searches every five steps
    add("forge_384k_mixed", "contact", 384000, 200, precision="mixed", yielding=True, thermal=True)
    # an ensemble of 64 specimens in one context, each with its own material, punches and friction
    add("batch_64_mixed", "batch", 64, 150, precision="mixed", yielding=True)
    # the headline billet before yield, mixed precision and FP64
    add("upset_976k_mixed", "billet", 976000, 400, precision="mixed", yielding=False)
    add("upset_976k_fp64", "billet", 976000, 100, precision="fp64", yielding=False)
    # and a harder blow on worked stock, yielding: a neighbour search every five steps
    add("flow_976k_mixed", "billet", 976000, 200, precision="mixed", yielding=True)
    return c


def _default(kind):
    d = dict(kind=kind, precision="fp64", yielding=True)
    if kind == "billet":
        d.update(scheme="leapfrog", adaptive=False)
    if kind == "contact":
        d.update(thermal=False)
    return d


def draw(rng):
    kind = rng.choice(("billet", "billet", "billet", "billet", "contact", "contact", "plate2d", "damage", "batch",
                       "adjoint"))
    lo, hi = {"billet": (1500, 1000000), "contact": (1500, 400000), "plate2d": (1500, 60000),
              "damage": (3000, 120000), "batch": (6, 64), "adjoint": (3000, 120000)}[kind]
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    c = dict(_default(kind), n=n)
    if kind in ("billet", "contact", "plate2d", "batch"):
        c["precision"] = "mixed" if kind == "batch" else rng.choice(("mixed", "mixed", "fp64"))
    if kind in ("billet", "contact"):
        c["yielding"] = rng.random() < 0.6
    if kind == "billet":
        c["scheme"] = rng.choice(("leapfrog", "leapfrog", "kickdrift"))
        c["adaptive"] = rng.random() < 0.25
    if kind == "contact":
        c["thermal"] = rng.random() < 0.6
    steps = rng.randint(50, 200)
    if kind in ("adjoint", "batch"):
        steps = rng.randint(10, 40)
    elif n > 150000:
        steps = rng.randint(30, 60) if c["precision"] == "fp64" else rng.randint(60, 120)
    c["steps"] = steps
    return c


# ---------------------------------------------------------------------------
# inputs

JC_FLOW_PL = 0.05  # plastic strain of worked stock


def _jc(mat, pl):
    return (mat["jc_A"] + mat["jc_B"] * pl ** mat["jc_n"])


def _pitch(volume, n):
    return (volume / n) ** (1.0 / 3.0)


def _case(case, seed):
    """The cases.Case of the inputs and its extra initial fields (dict): the
    plastic strain and yield stress of worked stock, the stresses of a flow."""
    kind, steps = case["kind"], case["steps"]
    extra = {}
    if kind == "billet":
        R, L = 30e-3, 60e-3
        dx = _pitch(math.pi * R * R * L, case["n"])
        # a blow of at most 20 m/s that shortens the billet by at most 0.15 % per pass, or slow loading
        dt = 0.4 * 1.2 * dx / cases.elastic(AL["E"], AL["nu"], AL["rho"])[2]
        v = -min(20.0, 1.5e-3 * L / (dt * steps)) if case["yielding"] else -0.1
        c = cases.cylinder_case("billet", R, L, dx, AL["rho"], AL["E"], AL["nu"], cases.JC_AL, steps=steps,
                                jitter=1e-3, seed=seed, v_top=v, T0=300.0)
        if case["adaptive"]:
            c.auto_ts = 1
        if case["yielding"]:
            extra = _worked(c, cases.JC_AL, JC_FLOW_PL)
    elif kind == "damage":
        R, L, v = 7.5e-3, 30e-3, -2.0
        dx = _pitch(math.pi * R * R * L, case["n"])
        c = cases.cylinder_case("damage", R, L, dx, AL["rho"], AL["E"], AL["nu"], cases.JC_AL, steps=steps,
                                jitter=1e-3, seed=seed, v_top=v, T0=300.0)
        z = c.x[:, 2]
        c.ids = np.where(z < z.min() + 2.5 * dx, 2, np.where(z > z.max() - 2.5 * dx, 3, 0)).astype(np.int32)
        c.damage = {0: (0.2, 0.3, -2.0, 0.01, 0.4)}
        extra = _flowing(c, cases.JC_AL, v)
    elif kind == "plate2d":
        dx = math.sqrt(30e-3 * 60e-3 / case["n"])
        c = cases.plate2d_case("plate", 30e-3, 60e-3, dx, AL["rho"], AL["E"], AL["nu"], cases.JC_AL, steps=steps,
                               jitter=1e-3, seed=seed, v_top=-1.0, T0=300.0)
        extra = _worked(c, cases.JC_AL, JC_FLOW_PL)
    elif kind == "contact":
        R, L, v = 15e-3, 30e-3, -5.0 if case["n"] > 50000 else -2.0
        dx = _pitch(math.pi * R * R * L, case["n"])
        c = cases.config3(steps=steps, dx=dx, R=R, L=L, dens=32, v_punch=v, seed=seed)
        _stand_off(c, 3 * steps * abs(v) * c.dt)
        c.thermal = c.pl_heating = bool(case["thermal"])
        rng = np.random.Generator(np.random.PCG64(seed + 1))
        z = c.x[:, 2]
        c.T = 300.0 + 80.0 * (z - z.min()) / L + rng.uniform(-1.0, 1.0, c.n)
        c.v = _ringing(c.x, np.zeros(c.n, dtype=np.int64), abs(v))
        if case["yielding"]:
            extra = _worked(c, cases.STEEL_JC, 0.02)
    elif kind == "batch":
        c = cases.config4(n_spec=case["n"], steps=max(steps, 1))
        rng = np.random.Generator(np.random.PCG64(seed))
        c.x = c.x + rng.uniform(-1e-3, 1e-3, c.x.shape) * c.meta["dx"]
        _stand_off(c, 3 * steps * 5.0 * c.dt)
        c.group_sums = (-1, 4096)
        c.v = _ringing(c.x, c.material, 5.0)
        extra = dict(pl_strain=np.full(c.n, 0.02), sigmay=c.sigmay * 1.5)
    elif kind == "adjoint":
        R, L, v = 15e-3, 30e-3, -1.0
        c = cases.config5_zone(steps=steps, dx=_pitch(math.pi * R * R * L, case["n"]), R=R, L=L, v_top=v, seed=seed)
        extra = _flowing(c, cases.STEEL_JC, v)
    else:
        raise ValueError(kind)
    return c, extra


def _stand_off(c, gap):
    """The punches `gap` further from the billet: a blow that is about to land."""
    for m, s in zip(c.meshes, (1.0, -1.0)):
        if "nodes" in m:
            m["nodes"] = m["nodes"] + np.array([0.0, 0.0, s * gap])
        else:
            m["p1"] = tuple(m["p1"][:2]) + (m["p1"][2] + s * gap,)
            m["p2"] = tuple(m["p2"][:2]) + (m["p2"][2] + s * gap,)


def _worked(c, mat, pl):
    return dict(pl_strain=np.full(c.n, pl), sigmay=np.full(c.n, _jc(mat, pl)))


def _ringing(x, body, v):
    """Bodies still ringing along z from the last blow, their ends moving at v."""
    z, w = x[:, 2], np.zeros_like(x)
    nb = int(body.max()) + 1
    lo, hi = np.full(nb, np.inf), np.full(nb, -np.inf)
    np.minimum.at(lo, body, z)
    np.maximum.at(hi, body, z)
    w[:, 2] = -v * np.sin(math.pi * ((z - lo[body]) / (hi - lo)[body] - 0.5))
    return w


def _flowing(c, mat, v_top):
    """A billet in the middle of its upsetting: uniaxial compression at the
    yield stress of the worked metal, in uniform plastic flow."""
    x = c.x
    z0, L = x[:, 2].min(), np.ptp(x[:, 2])
    rate = -v_top / L
    c.v = np.stack([0.5 * rate * x[:, 0], 0.5 * rate * x[:, 1], -rate * (x[:, 2] - z0)], axis=1)
    Y = _jc(mat, JC_FLOW_PL)
    m = c.materials[0]
    n = c.n
    sig = np.zeros((n, 9))
    sig[:, 8] = -Y
    dev = np.zeros((n, 9))
    dev[:, 0] = dev[:, 4] = Y / 3.0
    dev[:, 8] = -2.0 * Y / 3.0
    c.density = np.full(n, m["ref_density"] + (Y / 3.0) / m["Cs"] ** 2)
    return dict(pl_strain=np.full(n, JC_FLOW_PL), sigmay=np.full(n, Y), sigma=sig, shear=dev)


def prepare(case, seed):
    c, extra = _case(case, seed)
    mx = capi.MIXED if case["precision"] == "mixed" else capi.FP64
    s = cases.make_solver(c, precision=mx)
    for name, a in extra.items():
        s.set(name, a)
    if case["kind"] == "adjoint":
        Y, R = _jc(cases.STEEL_JC, JC_FLOW_PL), c.meta["R"]
        return dict(solver=s, target=np.full(case["steps"], 0.98 * Y * math.pi * R * R), scheme=capi.LEAPFROG,
                    steps=case["steps"], adjoint=True)
    scheme = capi.KICKDRIFT if case.get("scheme") == "kickdrift" else capi.LEAPFROG
    s.prepare(scheme)
    return dict(solver=s, scheme=scheme, steps=case["steps"], adjoint=False)


# ---------------------------------------------------------------------------
# one pass

RESULTS = ("Position", "Velocity", "Pressure", "Density", "Sigma", "Strain", "Strain_pl", "Sigma_eq", "Temperature",
           "Pl_Strain", "ps_en", "Displacement")


def run(state):
    s = state["solver"]
    if state["adjoint"]:
        loss, hist = s.adj_forward(state["target"], checkpoint_every=20, kind=capi.ADJ_ZONE, index=3, component=2)
        grad = s.adj_backward()
        out = dict(loss=loss, history=hist, grad=grad)
        for name in ("x", "v", "sigmay", "pl_strain"):
            out[name] = s.adj_field(name)
        s.adj_restore()
        return out
    s.step(state["steps"], state["scheme"])
    s.sync()
    f, iv = s.pack_xdmf()
    n = s.n
    out = {}
    for name in RESULTS:
        o, w = output.XDMF_FLOAT[name]
        out[name] = f[o * n:(o + w) * n]
    out.update({name: iv[o * n:(o + 1) * n] for name, o in output.XDMF_INT.items()})
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    """Per step: the state (x, v, displacement, density, deviatoric stress,
    strain, plastic strain, yield stress, with the thermal solver T) read and
    written once in FP64, the neighbour rows read once (2 bytes per entry),
    and each pair's terms (acceleration 60, density 20, rates 45
    operations) formed once; once per pass the output table.  A gradient costs
    at least the window twice (forward, and again for the reverse sweep) plus
    the reverse step, which reads and writes the state and its adjoint."""
    kind, steps = case["kind"], case["steps"]
    n = case["n"] * 12700 if kind == "batch" else case["n"]
    nb = 17.0 if kind == "plate2d" else 55.0
    state = 24 + (1 if case.get("thermal") else 0)
    bytes_step = n * (2 * 8.0 * state + 2.0 * nb)
    flops_step = n * (nb / 2 * 125.0 + 250.0)
    if case.get("thermal"):
        flops_step += n * nb / 2 * 12.0
    if kind == "adjoint":
        return {"bytes": 4.0 * steps * bytes_step, "flops": 4.0 * steps * flops_step}
    return {"bytes": steps * bytes_step + 268.0 * n, "flops": steps * flops_step}


# ---------------------------------------------------------------------------
# the same run in 64 bits, in plain torch

def exact(case, seed):
    """The Leapfrog billet of up to 50 thousand particles, restated over a flat list of
    directed pairs.  The pairs are those of the start: over these runs no
    distance comes near the radius (the lattice's shells lie 2 % and more off
    it and the billet deforms by under 0.3 %).  The other kinds: None."""
    if case["kind"] != "billet" or case["scheme"] != "leapfrog" or case["adaptive"] or case["n"] > 50000:
        return None
    c, extra = _case(case, seed)
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    T = lambda a: torch.tensor(np.asarray(a, dtype=np.float64), device=dev)  # noqa: E731
    x, m, rho = T(c.x), T(c.mass), T(c.density)
    n, h, dt, M = c.n, float(c.h[0]), c.dt, c.materials[0]
    zero = torch.zeros(n, 6, dtype=torch.float64, device=dev)
    v = T(c.v) if c.v is not None else torch.zeros(n, 3, dtype=torch.float64, device=dev)
    pick = torch.tensor([0, 4, 8, 1, 2, 5], device=dev)  # xx yy zz xy xz yz
    sig = T(extra["sigma"])[:, pick] if "sigma" in extra else zero.clone()
    S = T(extra["shear"])[:, pick] if "shear" in extra else zero.clone()
    sy = T(extra.get("sigmay", c.sigmay))
    pl = T(extra["pl_strain"]) if "pl_strain" in extra else torch.zeros(n, dtype=torch.float64, device=dev)
    strain, epl, u = zero.clone(), zero.clone(), torch.zeros_like(v)
    ii, jj = [], []
    for a in range(0, n, 1024):
        d = (x[a:a + 1024, None, :] - x[None, :, :]).square_().sum(-1)
        near = d <= (2.0 * h) ** 2
        p, q = torch.nonzero(near, as_tuple=True)
        p = p + a
        keep = p != q
        ii.append(p[keep])
        jj.append(q[keep])
    i, j = torch.cat(ii), torch.cat(jj)
    c5 = 1.0 / (math.pi * h ** 5)
    add = lambda t: torch.zeros((n,) + t.shape[1:], dtype=torch.float64, device=dev).index_add_(0, i, t)  # noqa: E731

    def grad_w():
        e = x[i] - x[j]
        r2 = e.square().sum(-1)
        q = r2.sqrt() / h
        g = torch.where(q < 1, c5 * (-3 + 2.25 * q), torch.where(q < 2, -0.75 * c5 * (2 - q) ** 2 / q, torch.zeros_like(q)))
        return e, r2, g

    def mul(t, e):  # symmetric t times e
        return torch.stack([t[:, 0] * e[:, 0] + t[:, 3] * e[:, 1] + t[:, 4] * e[:, 2],
                            t[:, 3] * e[:, 0] + t[:, 1] * e[:, 1] + t[:, 5] * e[:, 2],
                            t[:, 4] * e[:, 0] + t[:, 5] * e[:, 1] + t[:, 2] * e[:, 2]], 1)

    bcs = [(torch.tensor(c.ids == b["zone"], device=dev), T(b["value"])) for b in c.bcs]
    K6 = torch.tensor([1.0, 1.0, 1.0, 2.0, 2.0, 2.0], dtype=torch.float64, device=dev)
    for step in range(case["steps"]):
        e, r2, g = grad_w()
        t = sig / (rho * rho)[:, None]
        vd = ((v[i] - v[j]) * e).sum(-1)
        mu = h * vd / (r2 + 0.01 * h * h)
        pi = torch.where(vd < 0, (M["alpha"] * M["Cs"] * mu + M["beta"] * mu * mu) / (0.5 * (rho[i] + rho[j])), torch.zeros_like(mu))
        a = add((m[j] * g)[:, None] * (mul(t[i] + t[j], e) + pi[:, None] * e))
        v = v + a * (0.5 * dt if step == 0 else dt)
        for z, val in bcs:
            v = torch.where(z[:, None], val[None, :], v)
        vol = m / rho
        rho = rho + dt * rho * add(vol[j] * g * ((v[i] - v[j]) * e).sum(-1))
        x = x + v * dt
        u = u + v * dt
        e, r2, g = grad_w()
        w = v[i] - v[j]
        cp = ((m / rho)[j] * (-0.5) * g)[:, None]
        G = add((cp[:, :, None] * w[:, :, None] * e[:, None, :]).reshape(-1, 9)).reshape(n, 3, 3)
        D, W = G + G.transpose(1, 2), G - G.transpose(1, 2)
        sr = torch.stack([D[:, 0, 0], D[:, 1, 1], D[:, 2, 2], D[:, 0, 1], D[:, 0, 2], D[:, 1, 2]], 1)
        full = torch.stack([S[:, 0], S[:, 3], S[:, 4], S[:, 3], S[:, 1], S[:, 5], S[:, 4], S[:, 5], S[:, 2]], 1).reshape(n, 3, 3)
        J = full @ W.transpose(1, 2) + W @ full
        jt = torch.stack([J[:, 0, 0], J[:, 1, 1], J[:, 2, 2], J[:, 0, 1], J[:, 0, 2], J[:, 1, 2]], 1)
        d6 = sr.clone()
        d6[:, :3] -= sr[:, :3].sum(-1, keepdim=True) / 3.0
        S = S + dt * (2.0 * M["G"] * d6 + jt)
        eff = torch.sqrt(0.5 * ((sr[:, 0] - sr[:, 1]) ** 2 + (sr[:, 1] - sr[:, 2]) ** 2 + (sr[:, 2] - sr[:, 0]) ** 2)
                         + 3.0 * (sr[:, 3:] ** 2).sum(-1))
        trial = torch.sqrt(1.5 * (S * S * K6).sum(-1))
        S = S * torch.clamp(sy / trial, max=1.0)[:, None]
        rate = torch.where(eff > M["jc_eps0"], 1.0 + M["jc_C"] * torch.log(eff / M["jc_eps0"]), torch.ones_like(eff))
        sy = (M["jc_A"] + M["jc_B"] * pl ** M["jc_n"]) * rate
        dep = torch.where(trial > sy, (trial - sy) / (3.0 * M["G"]), torch.zeros_like(sy))
        pl = pl + dep
        P = M["P0"] + M["Cs"] ** 2 * (rho - M["ref_density"])
        sig = S.clone()
        sig[:, :3] -= P[:, None]
        f = (dep / sy)[:, None]
        tr = sig[:, :3].sum(-1, keepdim=True)
        epl = epl + torch.cat([f * (1.5 * sig[:, :3] - 0.5 * tr), 1.5 * f * sig[:, 3:]], 1)
        strain = strain + dt * sr
    order = torch.tensor([0, 1, 2, 3, 5, 4], device=dev)  # the tables' order: 00 11 22 01 12 02
    got = {"Position": x, "Velocity": v, "Pressure": P, "Density": rho, "Sigma": sig[:, order], "Strain": strain[:, order],
           "Strain_pl": epl[:, order], "Sigma_eq": torch.sqrt(1.5 * (S * S * K6).sum(-1)), "Temperature": T(c.T),
           "Pl_Strain": pl, "Displacement": u}
    return {k: got[k].reshape(-1) if k in got else None for k in RESULTS + tuple(output.XDMF_INT)}
