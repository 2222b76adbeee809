"""Contexts that share the device: two of some 400 tiles each, stepped side by
side from two host threads, give the fields of each alone (a sweep's
workgroups take tiles by their number only when all of the launch are
running, else in the order in which they start), and the SA model's sweeps
of the library's choice those of its hyperplane sweeps.  The same operations
on the same operands: equal bit for bit (tolerance 0)."""
import os
import threading

import numpy as np
import pytest

from aerocfd_amd import Solver
from tests.test_gpu_sa_sweep import build as sa_box
from tests.test_gpu_tile_sweep import box

pytestmark = pytest.mark.gpu

DIMS = [(20, 162, 162), (26, 170, 154)]


def make(dims, kernel):
    case = box(dims, 1)
    case.cfg.lusgs_kernel, case.cfg.batch_blocks = kernel, 1 if kernel == 2 else 0
    sol = Solver(case.cfg, case.dims, case.subfaces)
    case.upload(sol)
    sol.prepare()
    return sol


@pytest.mark.parametrize("kernels", [(0, 0), (1, 1), (2, 0), (1, 2)])
def test_side_by_side(kernels):
    print("test_side_by_side", kernels, flush=True)
    alone = []
    for d, k in zip(DIMS, kernels):
        sol = make(d, k)
        try:
            sol.step(12)
            alone.append(sol.download(1, "q"))
        finally:
            sol.close()
        assert np.isfinite(alone[-1]).all()
    sols = [make(d, k) for d, k in zip(DIMS, kernels)]
    errors = []

    def march(sol):
        try:
            for _ in range(4):
                sol.step(3)
        except Exception as e:  # reported by the test's thread
            errors.append(e)

    try:
        threads = [threading.Thread(target=march, args=(s,)) for s in sols]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        for sol, ref in zip(sols, alone):
            assert np.array_equal(sol.download(1, "q"), ref)
    finally:
        for s in sols:
            s.close()


@pytest.mark.parametrize("dims", [(5, 10, 11), (8, 18, 19), (12, 40, 33)])
def test_sa_by_ticket(dims):
    print("test_sa_by_ticket", dims, flush=True)
    out = []
    for switch in ("ACFD_LU_HYPERPLANES", None):  # None: lusgs_kernel 0, by ticket
        if switch:
            os.environ[switch] = "1"
        try:
            case = sa_box(dims)
            case.cfg.lusgs_kernel = 0
            sol = Solver(case.cfg, case.dims, case.subfaces)
        finally:
            if switch:
                os.environ.pop(switch)
        try:
            case.upload(sol)
            sol.run_stage("physical_bc")
            sol.run_stage("getpri")
            sol.prepare()
            sol.step(3)
            out.append(sol.download(1, "nut"))
        finally:
            sol.close()
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])
