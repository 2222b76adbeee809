"""A block's WENO3 + Roe residual in FP64 does not depend on what else its
context holds: the same block alone, beside unconnected blocks that take the
context through every run length of the j / k kernels (1, 4, 8, 16 nodes a
thread, from the context's nodes), in a batched step and in the stateless
routine.  Every face is the same operations on the same operands: equal bit
for bit (tolerance 0); and against the oracle norm-wise 1e-12."""
import numpy as np
import pytest

from aerocfd_amd import FlowConfig, Solver, cases
from aerocfd_amd import solver as S
from oracle import oracle as O
from tests.helpers import rel_l2, smooth_noise

pytestmark = pytest.mark.gpu

DIMS = (37, 41, 23)


def block():
    rng = np.random.default_rng(7)
    shp = DIMS[::-1]
    rho, u, v, w, p = (b + smooth_noise(shp, rng, 0.1) for b in (1.0, 0.3, 0.0, 0.1, 1.0 / (1.4 * 0.25)))
    q = cases.conservative(rho, u, v, w, p)
    r = cases.ranges_of(DIMS, cases.box_subfaces(*DIMS, [-10] * 6))
    dx, ij = cases.uniform_metrics(r, (0.03, 0.025, 0.04))[:2]
    return r, q, dx + 0.5 * rng.standard_normal(dx.shape), ij * (1 + 0.1 * rng.random(ij.shape))


def resident(beside, batch):
    """rhsi of the inviscid stage, and q after a step, of the block."""
    _, q, dx, ij = block()
    dims = [DIMS] + ([(beside,) * 3] if beside else [])
    cfg = FlowConfig(ma=0.5, iflag_solver=1, iflag_time=1, iflag_timeadvance=4, batch_blocks=batch, dt=1e-4)
    sol = Solver(cfg, dims, [cases.box_subfaces(*d, [-10] * 6) for d in dims])
    try:
        for name, a in (("q", q), ("dxidx", dx), ("inv_j", ij), ("dt", np.full(ij.shape, 1e-4))):
            sol.upload(1, name, a)
        sol.run_stage("inviscid")
        rhsi = sol.download(1, "rhsi")
        sol.step(1)
        return rhsi, sol.download(1, "q")
    finally:
        sol.close()


def test_same_in_every_context():
    r, q, dx, ij = block()
    alone = resident(0, 0)
    ref = O.inviscid(O.Ext.from_list(r), q, dx, ij, 1.4)
    assert np.all(rel_l2(alone[0], ref) <= 1e-12), rel_l2(alone[0], ref)
    stateless = S.inviscid_flux_1(FlowConfig(ma=0.5), r, q, dx, ij)
    assert np.array_equal(stateless, alone[0])
    for beside in (0, 45, 160, 320):
        for batch in (0, 1):
            print("test_same_in_every_context", beside, batch, flush=True)
            got = resident(beside, batch)
            for a, b, what in zip(got, alone, ("rhsi", "q")):
                assert np.array_equal(a, b), (beside, batch, what, (a != b).sum(), np.abs(a - b).max())
