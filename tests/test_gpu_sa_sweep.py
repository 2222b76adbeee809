"""The SA model's tile sweeps (in place, and over the sweep layout) against
its hyperplane sweeps: lines of a tile's width and a node more and less,
blocks of one tile and of several, steps that leave every remainder of the
operands' read-ahead.  A node's value is 12 FP64 operations on its
neighbours', of which at most three times the block's side lie in a row;
each passes on less than it takes: 12 * 3 * 30 * 1.1e-16 = 1.2e-13 of the
largest value, allowed 1e-12."""
import os

import numpy as np
import pytest

from aerocfd_amd import FlowConfig, Solver, cases
from tests.helpers import perturb_case

pytestmark = pytest.mark.gpu


def build(dims):
    cfg = FlowConfig(ma=0.5, re=2.0e4, iflag_solver=0, iflag_turbulence=2, iflag_time=0, cfl=0.8)
    case = cases.Case("sa_box", cfg, [dims], [cases.box_subfaces(*dims, (-10, -40, -20, -30, -50, -10))])
    h = (0.1, 0.1, 0.1)
    xyz = cases.node_coords(case.ranges[0], (1, 1, 1), h, (0, 0, 0))
    dxidx, inv_j, al, be, ga = cases.uniform_metrics(case.ranges[0], h)
    cases._common_fields(case, 0, cases.vortex_state(xyz * 10 - 5, cfg.ma), dxidx, inv_j, al, be, ga)
    case.fields[0].update(aalpha=al, bbeta=be, ggamma=ga)
    perturb_case(case, seed=sum(dims), sa=True)
    return case


def nut(dims, sweep, batch, hyperplanes):
    if hyperplanes:
        os.environ["ACFD_LU_HYPERPLANES"] = "1"
    try:
        case = build(dims)
        case.cfg.lusgs_kernel, case.cfg.batch_blocks = sweep, batch
        sol = Solver(case.cfg, case.dims, case.subfaces)
        try:
            case.upload(sol)
            sol.run_stage("physical_bc")
            sol.run_stage("getpri")
            sol.prepare()
            sol.step(3)
            return sol.download(1, "nut")
        finally:
            sol.close()
    finally:
        os.environ.pop("ACFD_LU_HYPERPLANES", None)


@pytest.mark.parametrize("dims", [(4, 4, 4), (5, 10, 11), (6, 9, 18), (7, 17, 12), (8, 18, 19), (9, 11, 27), (10, 26, 9),
                                  (31, 10, 10)])
def test_sa_sweep(dims):
    print("test_sa_sweep", dims, flush=True)
    ref = nut(dims, 0, 0, True)
    assert np.isfinite(ref).all()
    for sweep, batch in ((1, 0), (2, 0), (2, 1)):
        got = nut(dims, sweep, batch, False)
        err = np.abs(got - ref).max() / np.abs(ref).max()
        assert err <= 1e-12, (sweep, batch, err)
