"""Where downloads go: into pinned arrays (whole, and ending where the pinned
memory ends) without the copying threads, and from several contexts, one
after another and side by side, with one set of threads, which ends with
the last context.  Every value comes back bit for bit."""
import ctypes as C
import os
import threading

import numpy as np
import pytest
import torch

from aerocfd_amd import FlowConfig, Solver, _lib, cases
from aerocfd_amd.solver import FIELDS

pytestmark = pytest.mark.gpu

DIMS = (64, 64, 30)  # q: 4.9 MB


def threads():
    return len(os.listdir("/proc/self/task"))


def make(seed):
    sol = Solver(FlowConfig(iflag_solver=1), [DIMS], [cases.box_subfaces(*DIMS, [-10] * 6)])
    q = np.random.default_rng(seed).standard_normal(sol.shape(1, "q"))
    sol.upload(1, "q", q)
    sol.download(1, "dt")  # 1 MB: whatever the runtime itself starts for a copy
    return sol, q


def test_pinned():
    print("test_pinned", flush=True)
    sol, q = make(1)
    try:
        whole = torch.empty(q.size + 1000, dtype=torch.float64, pin_memory=True).numpy()
        before = threads()
        for at in (0, 1000):
            whole[:] = -1.0
            dst = whole[at:at + q.size]
            _lib.check(sol.lib.acfd_download(sol.h, C.c_int(1), C.c_int(FIELDS["q"][0]),
                                             dst.ctypes.data_as(C.POINTER(C.c_double))))
            assert np.array_equal(dst, q.ravel())
            assert (np.delete(whole, np.s_[at:at + q.size]) == -1.0).all()
        assert threads() == before
    finally:
        sol.close()


def test_contexts_share():
    print("test_contexts_share", flush=True)
    made = [make(s) for s in range(3)]
    try:
        before = threads()
        for _ in range(2):
            for sol, q in made:
                assert np.array_equal(sol.download(1, "q"), q)
        assert before < threads() <= before + 8

        bad = []

        def fetch(sol, q):
            for _ in range(20):
                if not np.array_equal(sol.download(1, "q"), q):
                    bad.append(1)

        work = [threading.Thread(target=fetch, args=m) for m in made]
        for t in work:
            t.start()
        for t in work:
            t.join()
        assert not bad and threads() <= before + 8
        for sol, _ in made[:2]:
            sol.close()
        assert np.array_equal(made[2][0].download(1, "q"), made[2][1])
    finally:
        for sol, _ in made:
            sol.close()
    assert threads() == before
    sol, q = make(5)
    try:
        assert np.array_equal(sol.download(1, "q"), q)
    finally:
        sol.close()
