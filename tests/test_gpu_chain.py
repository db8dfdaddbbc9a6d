"""The FP64 continuation of small fields in one launch (k_chains, teams of
workgroups) and the FP64 tail launch (k_tail64): whole runs against the
oracle, within 1e-9 relative at every point, at the sizes where they change
over (a row and its lists in LDS; a member's terms), with the smallest
fields, one and several branches, points outside the tree, and sweep caps
that end a step before, at and after its tail."""
import ctypes
import os
import threading

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
    (241, {}, dict(num_phi=16, num_branches=1)),
    (300, dict(rectangular=1), dict(num_phi=36, num_branches=3)),
    (700, {}, dict(num_phi=16, num_branches=2)),
    (1144, {}, dict(num_phi=4, num_branches=1)),       # the largest row that fits
    (1145, {}, dict(num_phi=4, num_branches=1)),       # the sweeps with k_tail64
    (400, {}, dict(num_phi=72, num_branches=18)),      # teams of one, 960 000 terms: the sweeps
    (300, {}, dict(num_phi=64, num_branches=16)),      # teams of two, 270 000 terms a member
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
    assert info["tail_launches"] == (2 * (np_ // (2 * nb)) if (n, nb) in ((1145, 1), (400, 18)) else 1)


@pytest.mark.parametrize("n,nb", [(1, 1), (17, 1), (100, 1), (137, 2), (240, 3), (60, 40), (1000, 1)])
@pytest.mark.parametrize("predictor", [0, 2])
def test_chains_without_teams_are_the_same_bits(workdir, n, nb, predictor):
    """members that give up at once: one workgroup per chain does their work,
    and the counts are those of one solve"""
    kw = dict(starfile=_stars(workdir, n), outfile_prefix="./", kappa_tot=0.45, shear=0.3, num_phi=8 * nb, num_branches=nb,
              predictor=predictor)
    with ccf_amd.Context(**kw) as c, ccf_amd.Context(**kw) as d:
        assert c.run(0), c.last_error()
        assert d.lib.ccf_set_team_wait(ctypes.c_void_p(d.ptr), ctypes.c_longlong(0)) == 0
        assert d.run(0) and d.run(0), d.last_error()
        assert np.array_equal(c.array(ccf_amd.ARRAY_CCS), d.array(ccf_amd.ARRAY_CCS))
        assert np.array_equal(c.array(ccf_amd.ARRAY_CAUSTICS), d.array(ccf_amd.ARRAY_CAUSTICS))
        a, b = c.info(), d.info()
    for k in ("points_converged", "points_total", "updates_full", "updates_early", "tail_sweeps", "flops_tail"):
        assert a[k] == b[k], k


def test_teams_of_several_contexts_at_once(workdir):
    """chains of contexts that run side by side from their own threads (teams
    of 32, 30 and 64 workgroups a launch) give the bits of each alone"""
    fields = [(100, 1), (400, 1), (137, 3), (240, 1)]
    kws = [dict(starfile=_stars(workdir, n), outfile_prefix="./", kappa_tot=0.45, shear=0.3, num_phi=40 * nb, num_branches=nb)
           for n, nb in fields]
    alone = []
    for kw in kws:
        with ccf_amd.Context(**kw) as c:
            assert c.run(0), c.last_error()
            alone.append(c.array(ccf_amd.ARRAY_CCS))
    got = [[] for _ in kws]
    start = threading.Barrier(len(kws))

    def work(k):
        with ccf_amd.Context(**kws[k]) as c:
            start.wait()
            for _ in range(3):
                got[k].append(c.array(ccf_amd.ARRAY_CCS) if c.run(0) else None)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(kws))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, a in enumerate(alone):
        assert len(got[k]) == 3 and all(np.array_equal(a, g) for g in got[k]), fields[k]


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


def test_error_pass_in_blocks_of_rows(workdir):
    """a phi grid of more rows than a launch of the error pass takes: the
    caustics it forms are the lens map of every row's roots"""
    sf = _stars(workdir, 17)
    with ccf_amd.Context(starfile=sf, outfile_prefix="./", kappa_tot=0.45, shear=0.3, num_phi=32780, num_branches=1) as c:
        assert c.run(0), c.last_error()
        z, w, info = c.array(ccf_amd.ARRAY_CCS).ravel(), c.array(ccf_amd.ARRAY_CAUSTICS).ravel(), c.info()
        e = c.eval_points(z, 0.0)
    assert info["points_converged"] == info["points_total"] == z.size
    g = e[:, 4] + 1j * e[:, 5]
    assert (np.abs(w - g) / np.maximum(np.abs(g), 1.0)).max() < 1e-11


@pytest.mark.parametrize("n,nb", [(17, 1), (100, 1), (137, 2), (240, 3), (1000, 1), (300, 16)])
def test_teams_meet(workdir, n, nb):
    """the teams of a run that has the device to itself meet, for every size
    of team; members that may not wait give up"""
    kw = dict(starfile=_stars(workdir, n), outfile_prefix="./", kappa_tot=0.45, shear=0.3, num_phi=8 * nb, num_branches=nb)
    with ccf_amd.Context(**kw) as c:
        for wait, retries in ((-1, 0), (0, 1), (-1, 0)):
            assert c.lib.ccf_set_team_wait(ctypes.c_void_p(c.ptr), ctypes.c_longlong(wait)) == 0
            assert c.run(0), c.last_error()
            assert c.lib.ccf_team_retries(c.ptr) == retries, wait
