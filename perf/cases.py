"""Timed cases of the critical-curve finder, through its public entry points.

Three kinds of work, each over the range in which it is used:

- ``run``: a whole field. One pass is ``Context.run`` (star file, tree and FMM
  build, Aberth solve at the branch centres, phi continuation, 1/mu error pass,
  caustic map) and the copies of the critical curves and caustics to the host,
  as a program that goes on with the curves makes them.
- ``batch``: several uneven fields solved together, ``Batch.run`` and the same
  arrays of every field.
- ``eval``, ``sweep``, ``root_sums``: the calls on a prepared field that take
  points or roots from the host: Witt's function, its derivative and the lens
  map at given points; one Aberth sweep; the root-sum FMM.

Star fields are synthetic: positions uniform in the disc or rectangle the field's
parameters give, masses equal or from a power law on [0.08, 1] (slope -2.35, or the
Kroupa slopes -1.3 and -2.3 with the break at 0.5), written in the reference's
star-file layout. The autotuner, whose choices follow from timings, is off: the same
field then gives the same bits.
"""
import os
import struct
import tempfile

import numpy as np
import torch

import ccf_amd

# the mixed-precision form as the benchmark runs it
MIXED = dict(precision=1, predictor=4, root_fmm=1)


def listed():
    return [
        # 100 equal masses, direct star sums, FP64: the smallest run, where launches and latency count
        dict(name="run 100 direct fp64", kind="run", num_stars=100, mass="equal", kappa=0.3, kappa_star=0.3, shear=0.1,
             num_phi=100, num_branches=1, direct=1),
        # the reference's default field: 137 equal masses with smooth matter, FP64
        dict(name="run 137 default fp64", kind="run", num_stars=137, mass="equal", kappa=0.3, kappa_star=0.27, shear=0.3,
             num_phi=100, num_branches=1),
        # 2000 stars, Salpeter, FMM order 20, FP64: an ordinary run over a fine phi grid
        dict(name="run 2000 fp64", kind="run", num_stars=2000, mass="salpeter", kappa=0.45, kappa_star=0.45, shear=0.35,
             num_phi=1000, num_branches=10, fmm_order=20),
        # 10 000 equal masses at the default phi grid, FP64: the run the reference published
        dict(name="run 10000 fp64", kind="run", num_stars=10000, mass="equal", kappa=0.4, kappa_star=0.4, shear=0.4,
             num_phi=100, num_branches=1),
        # the benchmark's field: 10 000 stars, Salpeter, order 24, 20 branches of 100 steps, mixed precision (the largest run)
        dict(name="run 10000 mixed", kind="run", num_stars=10000, mass="salpeter", kappa=0.5, kappa_star=0.5, shear=0.2,
             num_phi=2000, num_branches=20, fmm_order=24, mixed=1),
        # 50 000 stars, Kroupa, rectangular with smooth matter, order 28, mixed precision, on a coarser phi grid
        dict(name="run 50000 rect mixed", kind="run", num_stars=50000, mass="kroupa", kappa=0.7, kappa_star=0.35, shear=0.25,
             rectangular=1, num_phi=160, num_branches=8, fmm_order=28, mixed=1),
        # uneven fields of 50 to 1000 equal masses, num_phi 504 with 4 branches, FP64
        dict(name="batch 24 fp64", kind="batch", fields=24, stars_lo=50, stars_hi=1000, num_phi=504, num_branches=4),
        # such fields in mixed precision, more of them
        dict(name="batch 32 mixed", kind="batch", fields=32, stars_lo=50, stars_hi=1000, num_phi=504, num_branches=4, mixed=1),
        # f0, f1, w, length scale and 1/mu bound at host points of the 10 000-star field (a map of the field)
        dict(name="eval 100000 of 10000", kind="eval", num_stars=10000, mass="salpeter", kappa=0.5, kappa_star=0.5, shear=0.2,
             n=100000),
        # the same at a handful of points of a small field
        dict(name="eval 1000 of 100", kind="eval", num_stars=100, mass="equal", kappa=0.3, kappa_star=0.3, shear=0.1, n=1000),
        # one Aberth sweep over all roots of the 10 000-star field, FP64
        dict(name="sweep 20000 fp64", kind="sweep", num_stars=10000, mass="equal", kappa=0.4, kappa_star=0.4, shear=0.4, n=20000),
        # root sums of the 10 000-star field's roots by the FMM at its default order
        dict(name="root sums 20000", kind="root_sums", num_stars=10000, mass="salpeter", kappa=0.5, kappa_star=0.5, shear=0.2,
             n=20000),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case: sizes over the whole range (their logarithm), odd ones among them."""
    kind = rng.choice(["run", "run", "run", "batch", "eval", "sweep", "root_sums"])
    kappa_star = round(rng.uniform(0.1, 0.6), 3)
    smooth = rng.random() < 0.5
    c = dict(kind=kind, mass=rng.choice(["equal", "salpeter", "kroupa"]), kappa_star=kappa_star,
             kappa=round(kappa_star + (rng.uniform(0.02, 0.3) if smooth else 0.0), 3), shear=round(rng.uniform(0.0, 0.5), 3))
    if abs(1 - c["kappa"] - c["shear"]) < 0.05:
        c["shear"] = round(c["shear"] + 0.1, 3)  # away from a field of infinite magnification
    if kind == "run":
        c["mixed"] = int(rng.random() < 0.5)
        c["rectangular"] = int(rng.random() < 0.35)
        c["num_stars"] = _log_int(rng, 50, 30000 if c["mixed"] else 5000)
        c["num_branches"] = rng.choice([1, 2, 3, 5, 8])
        # the phi grid: a multiple of twice the branches, at most about 3 million points (1 million in FP64)
        most = (3e6 if c["mixed"] else 1e6) / (2 * c["num_stars"])
        steps = _log_int(rng, 6, max(8, min(400, int(most / (2 * c["num_branches"])))))
        c["num_phi"] = 2 * c["num_branches"] * steps
        if c["num_stars"] < 200 and rng.random() < 0.4:
            c["direct"] = 1
        if not c["rectangular"] and rng.random() < 0.2:
            c["approx"] = 0  # the disc's exact smooth sheet
    elif kind == "batch":
        c = dict(kind=kind, fields=rng.randint(3, 16), stars_lo=50, stars_hi=_log_int(rng, 100, 1000),
                 num_branches=rng.choice([1, 2, 4]), mixed=int(rng.random() < 0.5))
        c["num_phi"] = 2 * c["num_branches"] * rng.randint(10, 60)
    else:
        c["rectangular"] = int(rng.random() < 0.35)
        c["num_stars"] = _log_int(rng, 50, 20000)
        if kind == "eval":
            c["n"] = _log_int(rng, 200, 100000)
        else:
            c["n"] = _log_int(rng, 300, 20000)
            if kind == "sweep":
                c["mixed"] = int(rng.random() < 0.5)
    return c


def _masses(rng, mass, n):
    """n masses of unit-scale mass functions, scaled so that their mean is the function's: the field's size, and with
    it the number of roots of a rectangular one, does not depend on the seed"""
    if mass == "equal":
        return np.ones(n)
    # inverse CDF of a broken power law on [0.08, 1]
    pieces = [(0.08, 1.0, -2.35, 1.0)] if mass == "salpeter" else [(0.08, 0.5, -1.3, 1.0), (0.5, 1.0, -2.3, 0.5)]
    w = [b * (hi ** (s + 1) - lo ** (s + 1)) / (s + 1) for lo, hi, s, b in pieces]
    u = rng.random(n) * sum(w)
    out = np.empty(n)
    for (lo, hi, s, b), a, e in zip(pieces, np.cumsum([0.0] + w[:-1]), np.cumsum(w)):
        k = (u >= a) & (u <= e)
        out[k] = (lo ** (s + 1) + (u[k] - a) * (s + 1) / b) ** (1 / (s + 1))
    mean = sum(b * (hi ** (s + 2) - lo ** (s + 2)) / (s + 2) for lo, hi, s, b in pieces) / sum(w)
    return out * (n * mean / out.sum())


def _stars(c, seed):
    """(corner, n x 3 stars) of a field: the disc's radius or the rectangle's half sides from its surface density"""
    rng = np.random.default_rng(seed)
    n = c["num_stars"]
    m = _masses(rng, c["mass"], n)
    ax = np.array([1 / abs(1 - c["kappa"] + c["shear"]), 1 / abs(1 - c["kappa"] - c["shear"])])
    if c.get("rectangular"):
        corner = np.array([np.sqrt(ax[0] / ax[1]), np.sqrt(ax[1] / ax[0])]) * np.sqrt(np.pi * m.sum() / (4 * c["kappa_star"]))
        x = rng.uniform(-1, 1, (n, 2)) * corner
    else:
        corner = np.array([np.sqrt(m.sum() / c["kappa_star"]), 0.0])
        r, a = np.sqrt(rng.random(n)) * corner[0], 2 * np.pi * rng.random(n)
        x = np.stack([r * np.cos(a), r * np.sin(a)], axis=1)
    return corner, np.column_stack([x, m])


def _star_file(path, c, seed):
    corner, st = _stars(c, seed)
    with open(path, "wb") as f:
        f.write(struct.pack("<iiddd", len(st), 1 if c.get("rectangular") else 0, corner[0], corner[1], 1.0))
        f.write(np.ascontiguousarray(st, dtype="<f8").tobytes())


def _field_params(c, path, folder):
    # kappa_star of a file is its stars' own, equal to the field's to rounding
    p = dict(kappa_tot=c["kappa"] * (1 + 1e-12), shear=c["shear"], starfile=path, outfile_prefix=folder + os.sep)
    for k in ("num_phi", "num_branches", "fmm_order", "direct", "approx"):
        if k in c:
            p[k] = c[k]
    if c.get("mixed"):
        p.update(MIXED)
    return p


def _batch_fields(c, seed):
    """The fields of a batch: star counts spread evenly over their range (in no order), surface densities and shears
    uniform over theirs."""
    lo, hi, nf = c["stars_lo"], c["stars_hi"], c["fields"]
    counts = np.random.default_rng(nf).permutation(np.linspace(lo, hi, nf).round().astype(int))
    rng = np.random.default_rng(seed)
    out = []
    for i in range(c["fields"]):
        k = round(float(rng.uniform(0.1, 0.6)), 4)
        g = round(float(rng.uniform(0.0, 0.5)), 4)
        if abs(1 - k - g) < 0.05:
            g = round(g + 0.1, 4)
        out.append(dict(num_stars=int(counts[i]), mass="equal", kappa=k, kappa_star=k,
                        shear=g, num_phi=c["num_phi"], num_branches=c["num_branches"], mixed=c.get("mixed", 0)))
    return out


def _points(c, seed):
    """Host points of a prepared field: a map's points are uniform over it; roots lie near the
    stars, as the seeds of a solve do, and between them."""
    rng = np.random.default_rng([seed, 1])
    corner, st = _stars(c, seed)
    ext = corner if c.get("rectangular") else np.array([corner[0], corner[0]]) / np.sqrt(2)
    n = c["n"]
    z = (rng.uniform(-1, 1, (n, 2)) * ext).view(np.complex128).ravel()
    if c["kind"] != "eval":
        s = st[rng.integers(0, len(st), n // 2)]
        z[: n // 2] = s[:, 0] + 1j * s[:, 1] + rng.choice([-1.0, 1.0], n // 2) + 0.1 * rng.standard_normal((n // 2, 2)).view(np.complex128).ravel()
    return z


def prepare(case, seed):
    folder = tempfile.TemporaryDirectory()
    state = dict(case=case, folder=folder)
    if case["kind"] == "batch":
        b = ccf_amd.Batch()
        for i, f in enumerate(_batch_fields(case, seed)):
            path = os.path.join(folder.name, f"stars{i}.bin")
            _star_file(path, f, seed * 1000 + i)
            b.add(**_field_params(f, path, folder.name))
        state["batch"] = b
        return state
    path = os.path.join(folder.name, "stars.bin")
    _star_file(path, case, seed)
    ctx = ccf_amd.Context(**_field_params(case, path, folder.name))
    state["ctx"] = ctx
    if case["kind"] != "run":
        ctx.prepare()
        state["z"] = _points(case, seed)
        state["phi"] = float(np.random.default_rng([seed, 2]).uniform(0, 2 * np.pi))
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "batch":
        b = state["batch"]
        if not b.run(0):
            raise RuntimeError(b.last_error())
        n = range(len(b.params))
        return dict(ccs=[b.array(i, ccf_amd.ARRAY_CCS) for i in n], caustics=[b.array(i, ccf_amd.ARRAY_CAUSTICS) for i in n])
    c = state["ctx"]
    if kind == "run":
        if not c.run(0):
            raise RuntimeError(c.last_error())
        return dict(ccs=c.array(ccf_amd.ARRAY_CCS), caustics=c.array(ccf_amd.ARRAY_CAUSTICS))
    if kind == "eval":
        return c.eval_points(state["z"], state["phi"])
    if kind == "sweep":
        return c.aberth_sweep(state["z"], state["phi"])
    return c.root_sums(state["z"])


def _num_roots(c):
    return 2 * c["num_stars"]


def work(case):
    """Stars or points read once, results written once; per point one evaluation of the field (36 flops per star of
    a near field of about 40, 16 per expansion order of about 20), 10 per term of a sweep's direct sums."""
    if case["kind"] == "batch":
        mean = (case["stars_lo"] + case["stars_hi"]) / 2
        pts = case["fields"] * 2 * mean * (case["num_phi"] + case["num_branches"])
        return dict(bytes=24 * case["fields"] * mean + 32 * pts, flops=pts * (36 * 40 + 16 * 20))
    n = case["num_stars"]
    one = 36 * min(n, 40) + 16 * 20
    if case["kind"] == "run":
        pts = _num_roots(case) * (case["num_phi"] + case["num_branches"])
        return dict(bytes=24 * n + 32 * pts, flops=pts * one)
    if case["kind"] == "eval":
        return dict(bytes=24 * n + 80 * case["n"], flops=case["n"] * one)
    if case["kind"] == "sweep":
        return dict(bytes=24 * n + 32 * case["n"], flops=case["n"] * (one + 10 * (n + case["n"])))
    return dict(bytes=32 * case["n"], flops=case["n"] * 10 * 50)


def _sums(z, src, weight=None, powers=1):
    """sum over src of weight / (z - src)^k for k = 1 .. powers, the term at z itself left out"""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    zt, st = torch.from_numpy(z).to(dev), torch.from_numpy(src).to(dev)
    w = None if weight is None else torch.from_numpy(weight).to(dev)
    out = torch.zeros((powers, len(z)), dtype=torch.complex128, device=dev)
    step = max(1, int(4e7 / max(1, len(src))))
    for a in range(0, len(z), step):
        d = zt[a:a + step, None] - st[None, :]
        t = torch.where(d == 0, torch.zeros_like(d), 1 / d)
        p = t if w is None else t * w
        for k in range(powers):
            out[k, a:a + step] = p.sum(1)
            p = p * t
    return out.cpu().numpy()


def exact(case, seed):
    """The calls on a prepared disc field in 64 bits with every star and root summed directly. Whole runs have
    none (which index a root takes follows from the iteration), nor has the rectangle's smooth-sheet series."""
    kind = case["kind"]
    if kind in ("run", "batch"):
        return None
    z = _points(case, seed)
    if kind == "root_sums":
        return _sums(z, z)[0]
    if case.get("rectangular") or not case.get("approx", 1):
        return None
    _, st = _stars(case, seed)
    phi = float(np.random.default_rng([seed, 2]).uniform(0, 2 * np.pi))
    kappa = case["kappa"] * (1 + 1e-12)
    s = st[:, 0] + 1j * st[:, 1]
    s1, s2, s3 = _sums(z, s, st[:, 2], 3)
    a = 1 - kappa + case["kappa_star"]
    f0 = case["shear"] + s2 - a * np.exp(-1j * phi)
    f1 = -2 * s3
    if kind == "sweep":
        a0 = np.abs(f0)
        early = (np.abs(a0 * (a0 + 2 * a)) < 1e-9) & (np.abs(a0 * (a0 - 2 * a)) < 1e-9)
        pole = _sums(z, s)[0]
        return np.where(early, z, z - f0 / (f1 + f0 * (2 * pole - _sums(z, z)[0])))
    w = a * z + case["shear"] * z.conj() - s1.conj()
    dwb = case["shear"] + s2.conj()
    cct = -2j * dwb.conj() * (-2 * s3.conj())
    mu = 1 / (2 * np.abs(a * cct + dwb * cct.conj()))
    a0 = np.abs(f0)
    bound = np.maximum(np.abs(a0 * (a0 + 2 * a)), np.abs(a0 * (a0 - 2 * a)))
    return np.column_stack([f0.real, f0.imag, f1.real, f1.imag, w.real, w.imag, mu, bound])
