"""The pipelined tile sweep at the sizes where its tiling can go wrong:
blocks of 1 to 3 computed lines, lines around the 8 x 8 tile edge, more
tiles than fit on the device at once (handed out by ticket), against the
hyperplane sweeps of the same block.  Both schedules form every node from
the same expressions of the same operands, so the results are equal bit for
bit (tolerance 0)."""
import os
import sys

import numpy as np
import pytest

from aerocfd_amd import FlowConfig, Solver, cases
from tests.helpers import perturb_case

pytestmark = pytest.mark.gpu


def box(dims, solver):
    """One block of a uniform grid on [0,1]^3, three faces interfaces onto
    its own opposite faces, steps of a disturbed state."""
    ni, nj, nk = dims
    h = tuple(1.0 / (n - 1) for n in dims)
    cfg = FlowConfig(ma=0.3, re=1000.0, iflag_solver=solver, iflag_time=1, iflag_timeadvance=2,
                     dt=0.3 * min(h) / (1.0 + 1.0 / 0.3))
    d, subs, org = cases.split_box(ni, nj, nk, phys=(-10,) * 6, periodic=(False, True, False))
    case = cases.Case("box", cfg, d, subs)
    xyz = cases.node_coords(case.ranges[0], org[0][0], h, (0.0, 0.0, 0.0))
    one = np.ones_like(xyz[0])
    q = cases.conservative(one, one, 0.1 * one, -0.1 * one, one / (1.4 * 0.09))
    cases._common_fields(case, 0, q, *cases.uniform_metrics(case.ranges[0], h))
    return perturb_case(case, seed=sum(dims))


def run(case, kernel, batch=0, tickets=False):
    case.cfg.lusgs_kernel, case.cfg.batch_blocks = kernel, batch
    if tickets:
        os.environ["ACFD_LU_TICKETS"] = "1"
    if kernel == "hyperplanes":
        os.environ["ACFD_LU_HYPERPLANES"] = "1"
        case.cfg.lusgs_kernel = 0
    try:
        sol = Solver(case.cfg, case.dims, case.subfaces)
        try:
            case.upload(sol)
            sol.prepare()
            sol.step(3)
            return sol.download(1, "q"), sol.residual()
        finally:
            sol.close()
    finally:
        os.environ.pop("ACFD_LU_TICKETS", None)
        os.environ.pop("ACFD_LU_HYPERPLANES", None)


@pytest.mark.parametrize("solver", [0, 1])
@pytest.mark.parametrize("dims", [(4, 4, 4), (5, 5, 4), (4, 9, 12), (40, 10, 11), (12, 7, 17), (33, 18, 5),
                                  (9, 26, 25), (70, 8, 9)])
def test_tiles_equal_hyperplanes(dims, solver):
    print("test_tiles_equal_hyperplanes", dims, solver, flush=True)
    sys.stdout.flush()
    ref = run(box(dims, solver), "hyperplanes")
    assert np.isfinite(ref[0]).all()
    for kernel, batch, tickets in ((0, 0, False), (1, 0, False), (1, 0, True), (2, 1, False), (2, 0, True)):
        got = run(box(dims, solver), kernel, batch, tickets)
        assert np.array_equal(ref[0], got[0]), (dims, kernel, tickets, np.abs(ref[0] - got[0]).max())
        assert np.array_equal(ref[1], got[1])


def test_more_tiles_than_fit():
    """800 x 56 lines: 700 tiles of a short block (a device holds 512 or 256
    of the sweep's workgroups)."""
    dims = (8, 802, 58)
    print("test_more_tiles_than_fit", dims, flush=True)
    ref = run(box(dims, 1), "hyperplanes")
    got = run(box(dims, 1), 1)
    assert np.array_equal(ref[0], got[0])
