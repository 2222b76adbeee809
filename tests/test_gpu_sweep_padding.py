"""Blocks of one context do not reach each other through the tile sweeps'
workspace, which blocks swept one after another share: with every value of
one block NaN, an unconnected block of another size marches as it does alone,
and once the first block is written anew, as in a new context.  The same
operations on the same operands: equal bit for bit (tolerance 0)."""
import numpy as np
import pytest

from aerocfd_amd import FlowConfig, Solver, cases
from tests.helpers import perturb_case

pytestmark = pytest.mark.gpu


def boxes(dims, solver, kernel):
    """Unconnected blocks, every face farfield."""
    cfg = FlowConfig(ma=0.3, re=1000.0, iflag_solver=solver, iflag_time=1, iflag_timeadvance=2, lusgs_kernel=kernel,
                     batch_blocks=1 if kernel == 2 else 0, dt=2e-3)
    case = cases.Case("boxes", cfg, list(dims), [cases.box_subfaces(*d, [-10] * 6) for d in dims])
    for m, d in enumerate(dims):
        shp = (d[2], d[1], d[0])
        one = np.ones(shp)
        q = cases.conservative(one, one, 0.1 * one, -0.1 * one, one / (1.4 * 0.09))
        cases._common_fields(case, m, q, *cases.uniform_metrics(case.ranges[m], tuple(1.0 / (n - 1) for n in d)))
        one_block = cases.Case("box", cfg, [d], [case.subfaces[m]])
        one_block.fields[0] = case.fields[m]
        perturb_case(one_block, seed=sum(d))
    return case


def march(sol, case, sick=None):
    for m, fields in enumerate(case.fields):
        for name, a in fields.items():
            sol.upload(m + 1, name, np.full_like(a, np.nan) if m == sick and name == "q" else a)
    sol.run_stage("getpri")
    sol.prepare()
    sol.step(3)
    return [sol.download(m + 1, "q") for m in range(len(case.dims))]


@pytest.mark.parametrize("solver", [0, 1])
@pytest.mark.parametrize("kernel", [0, 1, 2])
@pytest.mark.parametrize("dims", [((12, 20, 11), (9, 13, 19)), ((9, 13, 19), (12, 20, 11)), ((30, 6, 5), (5, 21, 22))])
def test_blocks_apart(dims, kernel, solver):
    print("test_blocks_apart", dims, kernel, solver, flush=True)
    both = boxes(dims, solver, kernel)
    alone = []
    for m in range(2):
        one = boxes([dims[m]], solver, kernel)
        sol = Solver(one.cfg, one.dims, one.subfaces)
        try:
            alone.append(march(sol, one)[0])
        finally:
            sol.close()
        assert np.isfinite(alone[m]).all()
    sol = Solver(both.cfg, both.dims, both.subfaces)
    try:
        for sick in (0, 1, 0):
            got = march(sol, both, sick)
            assert np.isnan(got[sick]).any()
            assert np.array_equal(got[1 - sick], alone[1 - sick]), (sick, np.isnan(got[1 - sick]).sum())
            well = march(sol, both)
            for m in range(2):
                assert np.array_equal(well[m], alone[m]), (sick, m, np.isnan(well[m]).sum())
    finally:
        sol.close()
