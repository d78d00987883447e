"""Neighbour rows of small models, built by many lanes per particle, and of
those just above, by one: the pairs equal brute force exactly, and a row
that does not fit is reported."""
import numpy as np
import pytest

from weldform_amd import capi, cases

pytestmark = pytest.mark.gpu


def _case(n):
    """The first n particles of a jittered lattice, layer after layer."""
    rng = np.random.default_rng(n)
    k = np.arange(n)
    side = 24
    x = np.stack([k % side, k // side % side, k // side ** 2], axis=1) * 1.0e-3
    x = x + rng.uniform(-2e-4, 2e-4, (n, 3))
    c = cases.small_jc()
    c.x, c.h, c.mass, c.density = x, np.full(n, 1.2e-3), np.full(n, 2.7e-6), np.full(n, 2700.0)
    c.ids, c.material = np.zeros(n, dtype=np.int32), np.zeros(n, dtype=np.int32)
    c.sigmay, c.T = np.full(n, 1e8), np.full(n, 300.0)
    c.dom_max, c.dom_min = (0.03,) * 3, (-0.005,) * 3
    return c


def _brute(c):
    out = []
    for a in range(0, c.n, 1024):
        d = np.sqrt(((c.x[a:a + 1024, None, :] - c.x[None]) ** 2).sum(axis=2))
        i, j = np.nonzero(d / c.h[0] <= 2.0)
        i = i + a
        out.append(np.stack([i, j], axis=1)[i < j])
    return np.concatenate(out)


@pytest.mark.parametrize("precision", [capi.FP64, capi.MIXED])
@pytest.mark.parametrize("n", [1, 33, 577, 3001, 8192, 8193])
def test_rows_match_brute_force(n, precision):
    c = _case(n)
    print("n", n, "precision", precision, flush=True)
    s = cases.make_solver(c, precision=precision)
    s.rebuild_neighbours()
    got = s.neighbour_pairs()
    want = _brute(c)
    want = want[np.lexsort((want[:, 1], want[:, 0]))]
    assert np.array_equal(got, want)
    nb = np.bincount(want.ravel(), minlength=n)
    assert np.array_equal(s.get_int("nb"), nb)
    assert s.neighbour_stats() == (2 * len(want), nb.max())


@pytest.mark.parametrize("n", [577, 2048, 2049])
def test_rows_of_a_plate_match_brute_force(n):
    """Plane strain: many lanes per particle up to 2,048 particles."""
    rng = np.random.default_rng(n)
    k = np.arange(n)
    c = cases.plate2d_small(steps=1)
    c.x = np.stack([k % 48 * 1.0e-3, k // 48 * 1.0e-3, np.zeros(n)], axis=1)
    c.x[:, :2] += rng.uniform(-2e-4, 2e-4, (n, 2))
    for f in ("h", "mass", "density", "ids", "material", "sigmay", "T"):
        setattr(c, f, np.resize(getattr(c, f), n))
    print("n", n, flush=True)
    s = cases.make_solver(c)
    s.rebuild_neighbours()
    want = _brute(c)
    want = want[np.lexsort((want[:, 1], want[:, 0]))]
    assert np.array_equal(s.neighbour_pairs(), want)
    assert np.array_equal(s.get_int("nb"), np.bincount(want.ravel(), minlength=n))


@pytest.mark.parametrize("n", [3001, 8193])
def test_overfull_row_is_reported(n):
    s = cases.make_solver(_case(n), max_nb=40)
    with pytest.raises(capi.WFError) as e:
        s.rebuild_neighbours()
    assert e.value.code == capi.ENBOVERFLOW
