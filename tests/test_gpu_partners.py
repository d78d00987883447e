"""Contact partners of the free-surface particles, against brute force over
every rigid particle: counts equal exactly.  Rigid meshes fine against the
search cells give a particle hundreds of candidates, which whole wavefronts
walk; coarse ones a few, which the particle's own lane walks."""
import numpy as np
import pytest

from weldform_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dens,gap,scale", [(8, 1.0e-3, 1.0), (22, 1.1e-3, 1.0), (60, 1.33e-3, 1.0), (60, 1.33e-3, 2.2),
                                            (75, 1.3e-3, 1.0)])
def test_partner_counts(dens, gap, scale):
    """scale 2.2: 46k particles, the size class with a block per 128."""
    c = cases.contact_small(steps=1, dens=dens)
    if scale != 1.0:
        c = cases.config3(steps=1, dx=1.0e-3, R=7.5e-3 * scale, L=30e-3 * scale, dens=int(dens * scale), seed=5)
        c.thermal = c.pl_heating = False
    z = c.x[:, 2]
    for m, at in zip(c.meshes, (z.max() + gap, z.min() - gap)):
        m["p1"] = tuple(m["p1"][:2]) + (at,)
        m["p2"] = tuple(m["p2"][:2]) + (at,)
    s = cases.make_solver(c)
    nrig = sum(2 * m["dens"] ** 2 for m in c.meshes)
    print("n", c.n, "rigid", nrig, flush=True)
    xr = s.rigid("x", nrig)
    surf0 = s.get_int("id") == 1
    s.step(1)
    s.sync()
    got = s.get_int("contnb")
    both = surf0 & (s.get_int("id") == 1)
    hr = np.empty(nrig)
    e = 0
    for m in c.meshes:
        k = 2 * m["dens"] ** 2
        # a half square's radius: from its centroid to the far end of its legs
        leg = (m["p2"][0] - m["p1"][0]) / m["dens"]
        hr[e:e + k] = np.float32(1.1) * leg * np.sqrt(5.0) / 3.0
        e += k
    want = np.zeros(c.n, dtype=np.int64)
    margin = np.inf
    for i in np.flatnonzero(both):
        d = np.sqrt(((c.x[i] - xr) ** 2).sum(axis=1)) - (c.h[i] + hr)
        want[i] = (d < 0).sum()
        margin = min(margin, np.abs(d).min())
    print("largest count", want.max(), "pairs", want.sum(), "least margin", margin, flush=True)
    assert want.max() > 0 and margin > 1e-12
    assert np.array_equal(got, want)
