"""The calls on a prepared field that take points or roots from the host, at
the sizes where they change from the pinned buffer that the kernels read and
write to copies (eval 2048 points, sweeps and root sums 8192 roots), each
against the same call on pieces or the oracle's values."""
import numpy as np
import pytest

import ccf_amd
import oracle
from ccf_amd import io
from helpers import make_field

pytestmark = pytest.mark.gpu


def _points(sf, n, seed):
    _, _, corner, _, st = io.read_stars(sf)
    rng = np.random.default_rng(seed)
    z = 1.4 * abs(corner) * (rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n))  # some outside the tree
    return z


@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 2048, 2049, 70001])
def test_eval_sizes(workdir, n):
    sf = make_field(workdir, "salpeter300")
    kw = dict(kappa_tot=0.45, shear=0.35, num_phi=10)
    z = _points(sf, n, n)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", **kw) as c:
        c.prepare()
        g = c.eval_points(z, 1.1)
        assert np.array_equal(c.eval_points(z, 1.1), g)
        # a point's values do not depend on the points beside it
        k = max(0, n - 200)
        assert np.array_equal(c.eval_points(z[k:], 1.1), g[k:])
    o, _ = oracle.evaluate(oracle.params(starfile=sf, **kw), z[:3000], 1.1)
    for col in (0, 2, 4):
        a, b = g[:3000, col] + 1j * g[:3000, col + 1], o[:, col] + 1j * o[:, col + 1]
        assert (np.abs(a - b) / np.maximum(np.abs(b), 1.0)).max() < 1e-11


@pytest.mark.parametrize("n", [1, 8191, 8192, 8193])
@pytest.mark.parametrize("kw", [{}, dict(precision=1, root_fmm=1)])
def test_sweep_sizes(workdir, n, kw):
    sf = make_field(workdir, "salpeter300")
    z = _points(sf, n, 5)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", kappa_tot=0.45, shear=0.35, num_phi=10, **kw) as c:
        c.prepare()
        g = c.aberth_sweep(z, 0.7)
        assert np.all(np.isfinite(g)) and np.array_equal(c.aberth_sweep(z, 0.7), g)
        # the no-allocation sweep takes its row in by a copy
        assert np.array_equal(c.aberth_sweep_noalloc(z, 0.7), g)


@pytest.mark.parametrize("n", [1, 2, 8191, 8192, 8193])
def test_root_sum_sizes(workdir, n):
    sf = make_field(workdir, "salpeter300")
    z = _points(sf, n, 9)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", kappa_tot=0.45, shear=0.35, num_phi=10, root_fmm_order=14) as c:
        c.prepare()
        S = c.root_sums(z)
        assert np.array_equal(c.root_sums(z), S)
    pick = np.random.default_rng(1).choice(n, min(n, 300), replace=False)
    d = z[pick, None] - z[None, :]
    d[np.arange(pick.size), pick] = np.inf
    D, scale = (1 / d).sum(1), (1 / np.abs(d)).sum(1)
    # truncation at order 14 (3e-8 of the sum of moduli on uniform sets; the
    # bound that the 6000-root test of this order allows)
    assert np.all(np.abs(S[pick] - D) <= 2e-7 * scale)


def test_noalloc_sweep_largest_row(workdir):
    """the largest row that the no-allocation sweep's 32 MiB hold (mixed form, one root a thread)"""
    sf = make_field(workdir, "salpeter300")
    n = 194112
    z = _points(sf, n, 5)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", kappa_tot=0.45, shear=0.35, num_phi=10, precision=1, roots_per_thread=1) as c:
        c.prepare()
        g = c.aberth_sweep_noalloc(z, 0.7)
        assert np.array_equal(g, c.aberth_sweep(z, 0.7)) and np.any(g != z)
        with pytest.raises(RuntimeError, match="bytes of scratch"):
            c.aberth_sweep_noalloc(np.append(z, 0.5 + 0.5j), 0.7)
