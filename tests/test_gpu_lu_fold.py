"""A step whose viscous difference pass forms implicit1st's rhs and does the
unsteady find_dt, and whose halo fill and average1 share a launch, against
the same step taken stage by stage: the flow, rhs, rhsv (which
the step leaves out and a download forms), dt and its statistics are equal bit for bit."""
import numpy as np
import pytest

from aerocfd_amd import Solver, cases
from tests.test_gpu_parity import two_block_case

pytestmark = pytest.mark.gpu


def build(kind, precision):
    case = cases.tgv_box(21, blocks=((10,), (), (8,))) if kind == "tgv" else \
        two_block_case(ns=True, sa=kind.startswith("sa"), seed=5, itime=0 if kind.endswith("steady") else 1)
    case.cfg.precision = precision
    return case


def fields(sol, case):
    names = ("q", "rhs", "rhsv", "dt") + (("nut",) if case.cfg.iflag_turbulence == 2 else ())
    out = {(f, m): sol.download(m + 1, f) for m in range(len(case.dims)) for f in names}
    out["stats"] = sol.stats()
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("sweep,batch", [(1, 0), (2, 0), (1, 1), (2, 1)])
@pytest.mark.parametrize("kind", ["tgv", "ns", "ns_steady", "sa", "sa_steady"])
def test_fold(kind, sweep, batch, precision):
    print("test_fold", kind, sweep, batch, precision, flush=True)
    out = []
    for staged in (False, True):
        case = build(kind, precision)
        case.cfg.lusgs_kernel, case.cfg.batch_blocks = sweep, batch
        sol = Solver(case.cfg, case.dims, case.subfaces)
        try:
            case.upload(sol)
            sol.run_stage("physical_bc")
            sol.run_stage("getpri")
            sol.prepare()
            if staged:
                stages = ["getpri", "inviscid", "viscous", "find_dt", "implicit1st"] + \
                    (["sa"] if case.cfg.iflag_turbulence == 2 else []) + \
                    ["physical_bc", "update_buffer", "average", "getpri"]
                for _ in range(2):
                    for s in stages:
                        sol.run_stage(s)
            else:
                sol.step(2)
            out.append(fields(sol, case))
        finally:
            sol.close()
    for k in out[0]:
        assert np.isfinite(out[0][k]).all(), k
        assert np.array_equal(out[0][k], out[1][k]), (k, np.abs(out[0][k] - out[1][k]).max())
