"""The FP64 Cauchy sums with shared reciprocals (k_sums64_quad) through one
Aberth sweep, against the oracle's term-by-term sweep at the edges of the
kernel's tiles (64 listed roots), of its sparse form (at most 24) and of its
groups of four and 256 terms, and with roots beyond the range of a product of
four squared distances, which the kernel sums term by term."""
import numpy as np
import pytest

import ccf_amd
import oracle
from ccf_amd import io
from helpers import make_field

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _check(sf, roots, kw):
    phi = 2.1
    _, _, _, _, st = io.read_stars(sf)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", **kw) as c:
        c.prepare()
        g = c.aberth_sweep(roots, phi)
        assert np.array_equal(c.aberth_sweep_noalloc(roots, phi), g)
    o = oracle.aberth_sweep(oracle.params(starfile=sf, **kw), roots, phi)
    # the update is z - step, step = f0 / (f1 + f0 S): an error dS of the sums
    # moves it by step^2 dS. dS: a few roundings of every term, of the size of
    # the sum of the terms' moduli; f0 and f1 agree to about 1e-12.
    s = st[:, 0] + 1j * st[:, 1]
    scale = 2 * (1 / np.abs(roots[:, None] - s[None, :])).sum(1)
    for a in range(0, roots.size, 1024):
        d = np.abs(roots[a:a + 1024, None] - roots[None, :])
        d[d == 0] = np.inf
        scale[a:a + 1024] += (1 / d).sum(1)
    step = np.abs(o - roots)
    assert np.all(np.isfinite(g)) and step.max() > 0
    tol = 64 * EPS * (np.maximum(np.abs(roots), 1) + step * step * scale) + 1e-12 * step
    err = np.abs(g - o)
    assert np.all(err <= tol), (err / tol).max()


@pytest.mark.parametrize("n", [1, 2, 5, 24, 25, 63, 64, 65, 127, 255, 256, 257, 1030, 4101])
def test_quad_sums_at_tile_edges(workdir, n):
    sf = make_field(workdir, "cfg1")
    rng = np.random.default_rng(n)
    roots = 18 * (rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n))
    print(f"# quad sums, {n} roots", flush=True)
    _check(sf, roots, dict(kappa_tot=0.3, shear=0.1, direct=1, num_phi=10))


@pytest.mark.parametrize("n", [20, 300])
def test_quad_sums_far_roots(workdir, n):
    sf = make_field(workdir, "cfg1")
    rng = np.random.default_rng(n)
    roots = 18 * (rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n))
    roots[1], roots[2], roots[3] = 1e60, 2e60j, -3e59 + 1e59j
    print(f"# quad sums, {n} roots, three of them far off", flush=True)
    _check(sf, roots, dict(kappa_tot=0.3, shear=0.1, direct=1, num_phi=10))


@pytest.mark.parametrize("copies", [2, 5, 6, 8])
def test_quad_sums_coincident_roots(workdir, copies):
    """positions that coincide add nothing to each other's sums, also where a
    group's product of squared distances underflows"""
    sf = make_field(workdir, "cfg1")
    rng = np.random.default_rng(copies)
    roots = 18 * (rng.uniform(-1, 1, 48) + 1j * rng.uniform(-1, 1, 48))
    roots[8:8 + copies] = roots[8]
    phi, kw = 2.1, dict(kappa_tot=0.3, shear=0.1, direct=1, num_phi=10)
    _, _, _, _, st = io.read_stars(sf)
    s = st[:, 0] + 1j * st[:, 1]
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", **kw) as c:
        c.prepare()
        g = c.aberth_sweep(roots, phi)
        e = c.eval_points(roots, phi)
    f0, f1 = e[:, 0] + 1j * e[:, 1], e[:, 2] + 1j * e[:, 3]
    d = roots[:, None] - roots[None, :]
    t = np.where(d == 0, 0, 1 / np.where(d == 0, 1, d))
    u = 1 / (roots[:, None] - s[None, :])
    o = roots - f0 / (f1 + f0 * (2 * u.sum(1) - t.sum(1)))
    step = np.abs(o - roots)
    scale = 2 * np.abs(u).sum(1) + np.abs(t).sum(1)
    # (as in _check: roundings of the terms, and of f0 and f1)
    tol = 64 * EPS * (np.maximum(np.abs(roots), 1) + step * step * scale) + 1e-12 * step
    assert step.max() > 0 and np.all(np.abs(g - o) <= tol), (np.abs(g - o) / tol).max()


@pytest.mark.parametrize("n", [20, 30, 300])
@pytest.mark.parametrize("far", [1, 8])
def test_quad_sums_between_the_ranges(workdir, n, far):
    """roots so far off that a product of eight squared distances is out of
    range and one of four is not: the dense form's terms one by one, the
    sparse form's (at most 24 listed roots) in groups of four"""
    sf = make_field(workdir, "cfg1")
    rng = np.random.default_rng(n)
    roots = 18 * (rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n))
    roots[:far] = 1e25 * np.exp(0.7j * np.arange(1, far + 1)) * np.arange(1, far + 1)
    print(f"# quad sums, {n} roots, {far} of them far off", flush=True)
    _check(sf, roots, dict(kappa_tot=0.3, shear=0.1, direct=1, num_phi=10))
