"""The FP64 continuation of small fields in one launch (k_chains) and the FP64
tail launch (k_tail64): whole runs against the oracle, within 1e-9 relative
at every point, at the sizes where they change over (480 roots), with the
smallest fields, one and several branches, points outside the tree, and
sweep caps that end a step before, at and after its tail."""
import os

import numpy as np
import pytest

import ccf_amd
from ccf_amd import io
from helpers import compare_arrays, oracle_run

pytestmark = pytest.mark.gpu


def _stars(workdir, n, **kw):
    sf = os.path.join(str(workdir), f"chain_{n}_{kw.get('rectangular', 0)}.bin")
    if not os.path.exists(sf):
        ccf_amd.write_synthetic_stars(sf, 100 + n, num_stars=n, kappa_tot=0.45, kappa_star=0.4, shear=0.3,
                                      mass_function="salpeter", m_lower=0.08, m_upper=1.0, **kw)
    return sf


@pytest.mark.parametrize("n,field,grid", [
    (1, {}, dict(num_phi=20, num_branches=1)),
    (2, {}, dict(num_phi=12, num_branches=3)),
    (33, {}, dict(num_phi=24, num_branches=2)),
    (128, {}, dict(num_phi=20, num_branches=1, direct=1)),
    (64, dict(rectangular=1), dict(num_phi=24, num_branches=2)),
    (240, {}, dict(num_phi=16, num_branches=1)),       # the last rows of k_chains
    (241, {}, dict(num_phi=16, num_branches=1)),       # the first of the sweeps with k_tail64
    (300, dict(rectangular=1), dict(num_phi=36, num_branches=3)),
    (700, {}, dict(num_phi=16, num_branches=2)),
])
@pytest.mark.parametrize("predictor", [0, 3])
def test_fp64_continuation_matches_oracle(workdir, n, field, grid, predictor):
    sf = _stars(workdir, n, **field)
    kw = dict(kappa_tot=0.45, shear=0.3, **grid)
    print(f"# fp64 continuation, {n} stars {kw} predictor {predictor}", flush=True)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", predictor=predictor, **kw) as c:
        assert c.run(0), c.last_error()
        z, w, info = c.array(ccf_amd.ARRAY_CCS), c.array(ccf_amd.ARRAY_CAUSTICS), c.info()
    op = os.path.join(str(workdir), f"chain_{n}_{grid['num_phi']}_{grid['num_branches']}_{grid.get('direct', 0)}_")
    st = oracle_run(sf, op, **kw)
    R, nb, np_ = st["num_roots"], grid["num_branches"], grid["num_phi"]
    worst, nbad, bad = compare_arrays(z, io.read_array(op + "ccf_ccs.bin"), R, nb, details=True)
    if predictor == 0:
        assert nbad == 0, (worst, nbad)
        assert compare_arrays(w, io.read_array(op + "ccf_caustics.bin"), R, nb)[1] == 0
    else:
        # another path to each root: inside the 1/mu exit's band
        assert worst < 1e-6 and nbad <= max(5, 1e-3 * R * (np_ + nb)), (worst, nbad)
    assert info["points_converged"] == info["points_total"] == R * (np_ + nb)
    # one launch for the chains; else a tail for each step and side
    assert info["tail_launches"] == (1 if R <= 480 else 2 * (np_ // (2 * nb)))


@pytest.mark.parametrize("n", [100, 300])
@pytest.mark.parametrize("cap", [1, 2, 3])
def test_fp64_sweep_caps(workdir, n, cap):
    """step_iters bounds a step's sweeps in whichever kernel they run, and
    every point is written"""
    sf = _stars(workdir, n)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", kappa_tot=0.45, shear=0.3, num_phi=64, num_branches=1,
                         step_iters=cap) as c:
        assert c.run(0), c.last_error()
        z, info = c.array(ccf_amd.ARRAY_CCS), c.info()
    assert np.all(np.isfinite(z)) and np.all(z != 0)
    assert info["tail_sweeps"] <= 32 * 2 * cap
    assert info["updates_full"] + info["updates_early"] <= 2 * n * (60 + 64 * cap)
