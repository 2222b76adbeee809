"""The j / k inviscid kernels at every length of a thread's run (chosen from
the nodes: 1, 4, 8 for WENO3 + Roe in FP64; 2, 4 and 16 for the five-point
schemes), line lengths that leave a remainder, against the oracle: norm-wise
relative error at most 1e-12."""
import numpy as np
import pytest

from aerocfd_amd import FlowConfig, Solver, cases
from oracle import oracle as O
from tests.helpers import rel_l2, smooth_noise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,scheme", [(d, s) for d in [(10, 9, 8), (37, 5, 31), (130, 45, 19), (121, 102, 83)]
                                         for s in (0, 1, 2)] + [((170, 166, 150), 0)])
def test_runs(dims, scheme):
    print("test_runs", dims, scheme, flush=True)
    rng = np.random.default_rng(sum(dims))
    subs = cases.box_subfaces(*dims, [-10] * 6)
    h = tuple(1.0 / (n - 1) for n in dims)
    cfg = FlowConfig(ma=0.5, iflag_solver=1, inviscid_scheme=scheme,
                     iflag_timeadvance=2 if scheme == 0 else 4)
    r = cases.ranges_of(dims, subs)
    shp = (dims[2], dims[1], dims[0])
    rho, u, v, w, p = (b + smooth_noise(shp, rng, 0.1) for b in (1.0, 0.3, 0.0, 0.1, 1.0 / (1.4 * 0.25)))
    q = cases.conservative(rho, u, v, w, p)
    dx, ij = cases.uniform_metrics(r, h)[:2]
    sol = Solver(cfg, [dims], [subs])
    try:
        for k, a in (("q", q), ("dxidx", dx), ("inv_j", ij)):
            sol.upload(1, k, a)
        sol.run_stage("inviscid")
        got = sol.download(1, "rhsi")
    finally:
        sol.close()
    e = O.Ext.from_list(r)
    ref = O.inviscid(e, q, dx, ij, 1.4) if scheme == 0 else O.inviscid_ext(e, q, dx, ij, 1.4, scheme)
    assert np.all(rel_l2(got, ref) <= 1e-12), rel_l2(got, ref)
