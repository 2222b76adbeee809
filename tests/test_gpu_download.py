"""Downloads around the size at which the copying threads take over (2 MiB)
and around their chunks (1 MiB): every value of an uploaded field comes back
bit for bit, in new arrays and in a row."""
import numpy as np
import pytest

from aerocfd_amd import FlowConfig, Solver, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(64, 64, 12), (64, 64, 13), (64, 64, 64), (101, 67, 59), (41, 5, 4)])
def test_round_trip(dims):
    print("test_round_trip", dims, flush=True)
    sol = Solver(FlowConfig(iflag_solver=1), [dims], [cases.box_subfaces(*dims, [-10] * 6)])
    try:
        rng = np.random.default_rng(sum(dims))
        for _ in range(3):
            q = rng.standard_normal(sol.shape(1, "q"))
            met = rng.standard_normal(sol.shape(1, "dxidx"))
            sol.upload(1, "q", q)
            sol.upload(1, "dxidx", met)
            assert np.array_equal(sol.download(1, "q"), q)
            assert np.array_equal(sol.download(1, "dxidx"), met)
    finally:
        sol.close()
