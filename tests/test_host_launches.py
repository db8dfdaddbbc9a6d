"""What the host code asks of the device, on the CPU: a stand-in for the HIP
runtime (hip_stub.cpp) takes its place in a process of its own, runs no
kernel and writes down the launches, copies and synchronisations, which the
tests read back."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

FIELD = "kappa_tot=0.4, kappa_star=0.4, shear=0.2, direct=1, random_seed=3, outfile_prefix='./'"


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("stub") / "libhip_stub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", path, os.path.join(HERE, "hip_stub.cpp")], check=True)
    return path


def _log(stub, tmp_path, code):
    """the stand-in's lines for a program (Context and Batch of ccf_amd; `stub` the stand-in)"""
    log = str(tmp_path / "log")
    program = (f"import ctypes, sys\nstub = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)\nsys.path.insert(0, {ROOT!r})\n"
               f"import numpy as np\nimport ccf_amd\nstub.stub_log({log.encode()!r})\n" + code)
    r = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return [line.split() for line in open(log)]


def _launches(lines, kernel):
    """(grid x, y, z, workgroup) of a kernel's launches"""
    return [tuple(int(v) for v in w[2:6]) for w in lines if w[0] == "launch" and kernel in w[1]]


@pytest.mark.parametrize("num_phi,blocks", [(32766, 1), (32768, 2), (65600, 3)])
def test_error_pass_of_a_fine_phi_grid_fits_a_launch(stub, tmp_path, num_phi, blocks):
    """a launch holds 65 536 workgroups in y; the rows of a small field's run are num_phi + num_branches"""
    lines = _log(stub, tmp_path, f"c = ccf_amd.Context(num_stars=20, num_phi={num_phi}, num_branches=1, {FIELD})\nassert c.run(0)\n")
    assert _launches(lines, "k_chains")
    passes = _launches(lines, "k_errors")
    assert len(passes) == blocks and sum(g[1] for g in passes) == num_phi + 1
    assert all(int(v) <= 65536 for w in lines if w[0] == "launch" for v in w[3:5])


@pytest.mark.parametrize("kernel,n", [("k_batch_step_tail", 1), ("k_batch_sweep", 6), ("k_batch_step_tail", 4)])
def test_failed_batch_steps_leave_nothing_queued(stub, tmp_path, kernel, n):
    """an FP64 batch works on three streams; a launch that fails in between leaves all of them waited for, since the
    buffers that they use serve the next load"""
    lines = _log(stub, tmp_path, f"""
b = ccf_amd.Batch()
for stars in (300, 60, 320):
    b.add(num_stars=stars, num_phi=8, num_branches=1, {FIELD})
b.load(0)
b.build(0)
stub.stub_fail({kernel.encode()!r}, {n})
try:
    b.solve(0)
    raise SystemExit("the launch did not fail")
except RuntimeError:
    stub.stub_log(None)
assert b.run(0), b.last_error()
""")
    used = {}
    for k, w in enumerate(lines):
        if w[0] in ("launch", "sync"):
            used.setdefault(w[-1], {})[w[0]] = k
    assert sum("launch" in v for v in used.values()) == 3
    for s, v in used.items():
        assert v.get("sync", -1) > v.get("launch", -1), (s, lines[-5:])


@pytest.mark.parametrize("pinned", [False, True])
def test_copies_to_pinned_memory_go_there_at_once(stub, tmp_path, pinned):
    """one copy of the whole array to memory that the runtime knows; to other memory, copies into the slots"""
    lines = _log(stub, tmp_path, f"""
p = ctypes.c_void_p()
assert stub.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 23), 0) == 0
c = ccf_amd.Context(num_stars=100, num_phi=1000, num_branches=1, {FIELD})
assert c.run(0)
plain = np.empty(1 << 20)
base = (p.value if {pinned} else plain.ctypes.data) + 64
stub.stub_log({str(tmp_path / 'log').encode()!r})
r, k = ctypes.c_int(), ctypes.c_int()
assert c.lib.ccf_get_array(c.ptr, 1, ctypes.c_void_p(base), 1 << 22, ctypes.byref(r), ctypes.byref(k)) == 0
stub.stub_log(None)
""")
    copies = [int(w[1]) for w in lines if w[0] == "copy"]
    assert sum(copies) == 200 * 1001 * 16
    assert len(copies) == 1 if pinned else len(copies) > 1


def test_copy_slots_are_as_large_as_the_arrays_need(stub, tmp_path):
    """a program that makes a context for each field has the slots made and freed with each: one pinned allocation, for
    a small array at most twice its size; a larger one when a copy needs more, none when it needs less"""
    lines = _log(stub, tmp_path, f"""
def run(num_phi):
    c = ccf_amd.Context(num_stars=100, num_phi=num_phi, num_branches=1, {FIELD})
    assert c.run(0)
    return c
a, b, d = run(200), run(3000), run(50000)
stub.stub_log({str(tmp_path / 'log').encode()!r})
for c in (a, b, a, b, d, a, b, d):
    c.array(1)
stub.stub_log(None)
for c in (a, b, d):
    c.close()
""")
    pins = [int(w[1]) for w in lines if w[0] == "pin"]
    sizes = [200 * 201 * 16, 200 * 3001 * 16, 200 * 50001 * 16]
    assert len(pins) <= len(sizes) and pins == sorted(set(pins))
    assert pins[0] <= 2 * (sizes[0] + 4096) and pins[-1] <= 64 << 20
    assert len(pins) == 1 or pins[1] <= 2 * (sizes[1] + 8 * 4096)
    assert sum(w[0] == "unpin" for w in lines) == len(pins) - 1


@pytest.mark.parametrize("cus,branches,workgroups", [(256, 1, 24), (256, 4, 64), (256, 40, 80), (128, 1, 24), (128, 4, 32),
                                                     (32, 1, 8), (32, 4, 8), (32, 8, 16), (4, 1, 2)])
def test_teams_fit_a_quarter_of_the_device(stub, tmp_path, cus, branches, workgroups):
    """the workgroups that wait for each other are at most a quarter of the CUs (a member takes a whole one); with more
    rows than that none waits"""
    lines = _log(stub, tmp_path, f"""
stub.stub_cus({cus})
c = ccf_amd.Context(num_stars=50, num_phi={8 * branches}, num_branches={branches}, {FIELD})
assert c.run(0)
""")
    teams, alone = _launches(lines, "k_chains")
    assert teams[0] == workgroups and alone[0] == 2 * branches
    assert teams[0] <= max(cus // 4, 2 * branches)
