"""The hyperplane launches (ACFD_LU_HYPERPLANES=1) of contexts with several
blocks, uneven and rotated ones among them, with and without the SA model:
against the oracle, and as the other side of the tile sweeps (the library's
choice, per block, batched, both forms of q += dq), which form every node
from the same expressions of the same operands and so have to give the same
bits (tolerance 0).  That a Navier-Stokes run took the schedule it is named
for is read from the timers: a step forms rhs in a pass of its own for the
hyperplanes, and in the viscous pass for the tiles."""
import os

import numpy as np
import pytest

from aerocfd_amd import Solver, cases
from oracle import oracle as O
from tests.helpers import ora_config, ora_states, rel_l2
from tests.test_gpu_flat_plate import SMALL
from tests.test_gpu_parity import ROTATED_FLIP, ROTATED_PERM, two_block_case

pytestmark = pytest.mark.gpu

CUTS = ((6,), (6,), (6,))
CASES = {
    "tgv": lambda: cases.tgv_box(40),
    "tgv_8": lambda: cases.tgv_box(40, blocks=((20,), (16,), (24,))),
    "tgv_8_uneven": lambda: cases.tgv_box(33, blocks=((10,), (20,), (16,))),
    "vortex_12_uneven": lambda: cases.vortex_box(40, blocks=((13, 27), (17,), (9,))),
    "vortex_rotated": lambda: cases.vortex_box(12, blocks=CUTS, permute=ROTATED_PERM, flip=ROTATED_FLIP),
    "tgv_rotated": lambda: cases.tgv_box(12, blocks=CUTS, permute=ROTATED_PERM, flip=ROTATED_FLIP),
    "sa_two_block": lambda: two_block_case(ns=True, sa=True, seed=22, itime=0),
    "plate_12": lambda: cases.flat_plate(**SMALL),
}


def run(kind, nsteps, kernel, batch=0, env=()):
    """q (and nut) of every block, the residual norms, and the stages of one
    more implicit1st and SA update; kernel None: hyperplanes."""
    env = dict(env, ACFD_LU_HYPERPLANES="1") if kernel is None else dict(env)
    case = CASES[kind]()
    case.cfg.lusgs_kernel, case.cfg.batch_blocks = kernel or 0, batch
    sa = case.cfg.iflag_turbulence == 2
    os.environ.update(env)
    try:
        sol = Solver(case.cfg, case.dims, case.subfaces)
        try:
            case.upload(sol)
            sol.run_stage("physical_bc")
            sol.run_stage("getpri")
            sol.prepare()
            sol.step(nsteps - 1)
            sol.timing(True)
            sol.step(1)
            own_pass = sol.timing(False)["lusgs_other"][1] > 0
            assert case.cfg.iflag_solver == 1 or own_pass == (kernel is None), (kind, kernel, own_pass)
            names = ["q"] + (["nut"] if sa else [])
            out = [sol.download(m + 1, f) for m in range(len(case.dims)) for f in names]
            out.append(sol.residual())
            sol.run_stage("implicit1st")
            if sa:
                sol.run_stage("sa")
            out += [sol.download(m + 1, f) for m in range(len(case.dims)) for f in names]
            return out
        finally:
            sol.close()
    finally:
        for k in env:
            os.environ.pop(k, None)


@pytest.mark.parametrize("kind", sorted(CASES))
def test_tiles_equal_hyperplanes(kind):
    nsteps = 4
    ref = run(kind, nsteps, None)
    assert all(np.isfinite(a).all() for a in ref)
    for kernel, batch, env in ((0, 0, {}), (1, 0, {}), (1, 0, {"ACFD_LU_FUSED_ADD": "0"}), (0, 1, {}), (2, 0, {}),
                               (2, 1, {}), (2, 1, {"ACFD_LU_FUSED_ADD": "1"}), (2, 1, {"ACFD_LU_TICKETS": "1"})):
        print("test_tiles_equal_hyperplanes", kind, kernel, batch, env, flush=True)
        got = run(kind, nsteps, kernel, batch, env)
        for x, (a, b) in enumerate(zip(ref, got)):
            assert np.array_equal(a, b), (kernel, batch, env, x, np.abs(a - b).max())


@pytest.mark.parametrize("kind", ["vortex_rotated", "tgv_rotated", "plate_12"])
def test_hyperplanes_oracle(kind):
    """Ten steps: norm-wise relative error at most 1e-10, as the whole-step
    parity tests have it."""
    print("test_hyperplanes_oracle", kind, flush=True)
    nsteps = 10
    got = run(kind, nsteps, None)
    case = CASES[kind]()
    sa = case.cfg.iflag_turbulence == 2
    cfg = ora_config(case.cfg, case.totalnodes)
    states = ora_states(case)
    O.physical_bc(states, cfg)
    for st in states:
        st["pri_v"] = O.getpri(st.ext, st["q"], cfg.gamma, cfg.cv)[0]
    O.prepare(states, cfg)
    for _ in range(nsteps):
        O.step(states, cfg)
    per = 2 if sa else 1
    for m, st in enumerate(states):
        assert np.all(rel_l2(got[per * m], st["q"]) <= 1e-10), (m, rel_l2(got[per * m], st["q"]))
        if sa:
            assert rel_l2(got[per * m + 1], st["nut"]) <= 1e-10, m
