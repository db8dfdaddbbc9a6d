"""Large arrays to host memory through the pinned slots: copies made at the
same time from several threads and contexts (one of them holds the slots, the
others go through the runtime's own copy) give the same bytes, for sizes at
and around the slots' boundaries."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import ccf_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,num_phi,nb", [
    (64, 124, 2),     # 126 x 128 points: 258 048 B, just below the slots' smallest array
    (64, 128, 1),     # 129 x 128 points: 264 192 B, one part
    (64, 512, 1),     # 513 x 128 points: 1 050 624 B, two parts
    (64, 2046, 1),    # 2047 x 128 points: 4 192 256 B, seven parts
    (64, 2048, 2),    # 2050 x 128 points: 4 198 400 B, eight parts
    (137, 2000, 4),   # 8.8 MB, odd parts
    (700, 1200, 6),   # 27 MB, more parts than threads
    (700, 6000, 6),   # 134.5 MB: whole chunks
])
def test_concurrent_copies_agree(n, num_phi, nb):
    kw = dict(num_stars=n, kappa_tot=0.4, kappa_star=0.4, shear=0.2, num_phi=num_phi, num_branches=nb, random_seed=7,
              outfile_prefix="./")
    with ccf_amd.Context(**kw) as a, ccf_amd.Context(**kw) as b:
        assert a.run(0) and b.run(0)
        one = a.array(ccf_amd.ARRAY_CCS)
        got = {}
        start = threading.Barrier(4)

        def read(k, c, which):
            start.wait()
            got[k] = c.array(which)

        jobs = [(0, a, ccf_amd.ARRAY_CCS), (1, b, ccf_amd.ARRAY_CCS), (2, a, ccf_amd.ARRAY_CAUSTICS), (3, b, ccf_amd.ARRAY_CAUSTICS)]
        threads = [threading.Thread(target=read, args=j) for j in jobs]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert one.shape == (2 * n * nb, num_phi // nb + 1) and np.all(np.isfinite(one)) and np.all(one != 0)
    assert np.array_equal(got[0], one) and np.array_equal(got[1], one)
    assert np.array_equal(got[2], got[3]) and not np.array_equal(got[2], one)
    # a further context after the last one was destroyed (the slots were given back)
    with ccf_amd.Context(**kw) as c:
        assert c.run(0)
        assert np.array_equal(c.array(ccf_amd.ARRAY_CCS), one)


@pytest.mark.parametrize("offset", [0, 24])
def test_copy_to_pinned_memory(offset):
    """a destination that the runtime knows takes one copy, and the same bytes"""
    buf = torch.empty(1 << 21, dtype=torch.float64, pin_memory=True)
    with ccf_amd.Context(num_stars=137, kappa_tot=0.4, kappa_star=0.4, shear=0.2, num_phi=2000, num_branches=4, random_seed=7,
                         outfile_prefix="./") as c:
        assert c.run(0)
        one = c.array(ccf_amd.ARRAY_CCS)
        rows, cols = ctypes.c_int(), ctypes.c_int()
        assert c.lib.ccf_get_array(c.ptr, ccf_amd.ARRAY_CCS, ctypes.c_void_p(buf.data_ptr() + 8 * offset), 8 * (buf.numel() - offset),
                                   ctypes.byref(rows), ctypes.byref(cols)) == 0
    got = buf[offset:offset + 2 * one.size].numpy().view(np.complex128)
    assert one.nbytes >= 1 << 18 and np.array_equal(got, one.ravel())
