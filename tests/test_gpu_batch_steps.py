"""The FP64 phi steps that a batch's larger fields take together
(k_batch_sweep, k_batch_step_tail): whole batches against the oracle, within
1e-9 relative at every point, at the sizes where the rows change over from a
chain per workgroup (480 roots), with groups of 64 roots that are not full,
one and several branches, sweep caps that end a step before, at and after its
tail, and rows that do not fit a workgroup's LDS."""
import os

import numpy as np
import pytest

import ccf_amd
from ccf_amd import io
from helpers import compare_arrays, oracle_run

pytestmark = pytest.mark.gpu

KW = dict(kappa_tot=0.45, shear=0.3)


def _stars(workdir, n, **kw):
    sf = os.path.join(str(workdir), f"steps_{n}_{kw.get('rectangular', 0)}.bin")
    if not os.path.exists(sf):
        ccf_amd.write_synthetic_stars(sf, 300 + n, num_stars=n, kappa_tot=0.45, kappa_star=0.4, shear=0.3,
                                      mass_function="salpeter", m_lower=0.08, m_upper=1.0, **kw)
    return sf


@pytest.mark.parametrize("grid,predictor", [(dict(num_phi=20, num_branches=1), 0), (dict(num_phi=24, num_branches=3), 0),
                                            (dict(num_phi=36, num_branches=2), 3)])
def test_fp64_batch_steps_match_oracle(workdir, grid, predictor):
    fields = [(240, {}), (241, {}), (257, {}), (300, dict(rectangular=1)), (700, {})]
    b = ccf_amd.Batch()
    for n, f in fields:
        b.add(starfile=_stars(workdir, n, **f), outfile_prefix="./", fmm_order=20, predictor=predictor, **KW, **grid)
    assert b.run(0), b.last_error()
    first = [b.array(i, ccf_amd.ARRAY_CCS) for i in range(len(fields))]
    # a second solve gives the same bits
    b.solve(0)
    nb, np_ = grid["num_branches"], grid["num_phi"]
    for i, (n, f) in enumerate(fields):
        print(f"# field of {n} stars {f} {grid}", flush=True)
        z = b.array(i, ccf_amd.ARRAY_CCS)
        assert np.array_equal(z, first[i])
        op = os.path.join(str(workdir), f"steps_{n}_{np_}_")
        st = oracle_run(_stars(workdir, n, **f), op, fmm_order=20, **KW, **grid)
        R = st["num_roots"]
        worst, nbad, _ = compare_arrays(z, io.read_array(op + "ccf_ccs.bin"), R, nb, details=True)
        info = b.info(i)
        assert info["points_converged"] == info["points_total"] == R * (np_ + nb)
        if predictor == 0:
            assert nbad == 0, (n, worst, nbad)
            assert compare_arrays(b.array(i, ccf_amd.ARRAY_CAUSTICS), io.read_array(op + "ccf_caustics.bin"), R, nb)[1] == 0
        else:
            # another path to each root: inside the 1/mu exit's band
            assert worst < 1e-6 and nbad <= max(5, 1e-3 * R * (np_ + nb)), (n, worst, nbad)
    # a field's results do not depend on the batch around it
    alone = ccf_amd.Batch()
    n, f = fields[2]
    alone.add(starfile=_stars(workdir, n, **f), outfile_prefix="./", fmm_order=20, predictor=predictor, **KW, **grid)
    assert alone.run(0), alone.last_error()
    assert np.array_equal(alone.array(0, ccf_amd.ARRAY_CCS), first[2])
    b.close()
    alone.close()


@pytest.mark.parametrize("cap", [1, 2, 3, 4, 5])
def test_fp64_batch_sweep_caps(workdir, cap):
    """step_iters bounds a step's sweeps in whichever kernel they run, and
    every point is written"""
    n = 300
    b = ccf_amd.Batch()
    b.add(starfile=_stars(workdir, n), outfile_prefix="./", num_phi=16, num_branches=2, step_iters=cap, **KW)
    assert b.run(0), b.last_error()
    z, info = b.array(0, ccf_amd.ARRAY_CCS), b.info(0)
    assert np.all(np.isfinite(z)) and np.all(z != 0)
    rows = 16
    assert info["sweeps"] <= 2 * 60 + rows * cap
    assert info["updates_full"] + info["updates_early"] <= 2 * n * (2 * 60 + rows * cap)
    b.close()


def test_fp64_batch_rows_beyond_lds(workdir):
    """rows that do not fit a workgroup's LDS: the same root sets as the
    single-field path"""
    n, grid = 5000, dict(num_phi=16, num_branches=1)
    sf = _stars(workdir, n)
    b = ccf_amd.Batch()
    b.add(starfile=sf, outfile_prefix="./", fmm_order=20, **KW, **grid)
    assert b.run(0), b.last_error()
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", fmm_order=20, **KW, **grid) as c:
        assert c.run(0), c.last_error()
        s, R = c.array(ccf_amd.ARRAY_CCS), c.info()["num_roots"]
    worst, nbad = compare_arrays(b.array(0, ccf_amd.ARRAY_CCS), s, R, 1)
    assert nbad == 0, (worst, nbad)
    b.close()
