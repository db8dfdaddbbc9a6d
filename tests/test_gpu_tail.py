"""The mixed continuation on coarse phi grids, whose steps leave most of a
row active after their first sweep: their later sweeps run over the whole
device (k_witt with one evaluation, k_sums32_tail) until the rows are small
enough for k_tail. Against the oracle's run, with the same allowance as the
other mixed runs: a root may stop within twice the oracle's own Newton step
|f0/f1| of its root."""
import os

import numpy as np
import pytest

import ccf_amd
import oracle
from ccf_amd import io
from helpers import compare_arrays, newton_step, oracle_run

pytestmark = pytest.mark.gpu

FIELD = dict(num_stars=700, kappa_tot=0.45, kappa_star=0.4, shear=0.3, mass_function="salpeter", m_lower=0.08, m_upper=1.0)


def _stars(workdir):
    sf = os.path.join(str(workdir), "tail700.bin")
    if not os.path.exists(sf):
        ccf_amd.write_synthetic_stars(sf, 17, **FIELD)
    return sf


@pytest.mark.parametrize("grid,gkw", [
    (dict(num_phi=24, num_branches=1), dict(predictor=4, root_fmm=1)),
    (dict(num_phi=36, num_branches=3), dict(predictor=2)),
    (dict(num_phi=24, num_branches=2, direct=1), dict(predictor=4)),
])
def test_mixed_coarse_grid_matches_oracle(workdir, grid, gkw):
    sf = _stars(workdir)
    kw = dict(kappa_tot=0.45, shear=0.3, **grid)
    print(f"# mixed coarse grid {kw} {gkw}", flush=True)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", precision=1, **kw, **gkw) as c:
        assert c.run(0), c.last_error()
        got, info = c.array(ccf_amd.ARRAY_CCS), c.info()
    op = os.path.join(str(workdir), f"tail_{grid['num_phi']}_{grid['num_branches']}_")
    st = oracle_run(sf, op, **kw)
    R, nb, np_ = st["num_roots"], grid["num_branches"], grid["num_phi"]
    ref = io.read_array(op + "ccf_ccs.bin")
    worst, nbad, bad = compare_arrays(got, ref, R, nb, details=True)
    allowed = 2 * newton_step(sf, bad, np_, nb, **{k: v for k, v in kw.items() if k not in ("num_phi", "num_branches")})
    over = [(b, a) for b, a in zip(bad, allowed) if b[3] > 1e-9 * max(abs(b[2]), 1) + a]
    assert not over, over[:5]
    assert nbad <= max(5, 1e-3 * R * (np_ + nb)), nbad
    assert info["points_converged"] == info["points_total"] == R * (np_ + nb)
    # every step ended in a tail launch, after more than its first sweeps
    groups = min(2, nb)
    assert info["tail_launches"] == groups * np_ // (2 * nb)


@pytest.mark.parametrize("cap", [1, 2, 3])
def test_mixed_coarse_grid_sweep_caps(workdir, cap):
    """a cap on a step's sweeps that ends it before, at or after its tail:
    every point is written (finite), and a step runs no more sweeps"""
    sf = _stars(workdir)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", precision=1, predictor=4, kappa_tot=0.45, shear=0.3, num_phi=24,
                         num_branches=2, step_iters=cap) as c:
        assert c.run(0), c.last_error()
        z, info = c.array(ccf_amd.ARRAY_CCS), c.info()
    assert np.all(np.isfinite(z)) and np.all(z != 0)
    assert info["points_total"] == 1400 * 26
    # two groups of one branch, two rows each
    assert info["tail_sweeps"] <= 6 * 4 * (cap - 1)
