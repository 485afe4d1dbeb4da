"""The CM11a solver's one-workgroup tail and its sweeps per launch, at lattices
that put the edge of either somewhere else: no level below the finest fits it
or every one does, rows of odd padded length, axes that do not coarsen, lattices
narrower than a sweep tile, and one sweep more or less than the default.  Bar:
bit-exact against the CPU restatement."""
import numpy as np
import pytest

from test_oracle_cm11a import separating

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,sweeps", [((4, 4, 4), 6), ((8, 8, 8), 1), ((16, 16, 16), 6), ((20, 12, 12), 7),
                                         ((6, 6, 96), 2), ((48, 24, 12), 3), ((16, 64, 32), 5), ((64, 16, 32), 6)])
@pytest.mark.parametrize("open_top", [0, 1])
def test_levels_bit_exact(fpl, oracle, dims, sweeps, open_top):
    phi, u, v, w, h, dt, rho = separating(dims)
    P, (ou, ov, ow), orep = oracle.cm11a_project(phi, u, v, w, h, dt, rho, open_top=open_top, pre=sweeps, post=sweeps)
    g = fpl.UniformPressureProjection(dims, h)
    try:
        for _ in range(2):  # again on the same grid: no state carries over
            r = g.project(phi, u, v, w, dt, rho, solver="cm11a", open_top=open_top, lcp_sweeps=sweeps)
            assert np.array_equal(r.pressure, np.where(phi < 0, P[1:-1, 1:-1, 1:-1], 0))
            assert np.array_equal(r.u, ou) and np.array_equal(r.v, ov) and np.array_equal(r.w, ow)
            assert np.float32(r.report["lcp_residual"]) == np.float32(orep["lcp_residual"])
            assert r.report["coarse_sweeps"] == orep["coarse_sweeps"]
    finally:
        g.destroy()


def test_two_grids_alive(fpl):
    """A second grid whose tail is smaller leaves the first one's launches as they were."""
    scenes = [separating(d) for d in ((64, 64, 64), (16, 16, 16))]
    grids = [fpl.UniformPressureProjection(s[0].shape, s[4]) for s in scenes]
    try:
        first, second = [], []
        for out in (first, second):
            for g, (phi, u, v, w, h, dt, rho) in zip(grids, scenes):
                out.append(g.project(phi, u, v, w, dt, rho, solver="cm11a"))
        for a, b in zip(first, second):
            assert np.array_equal(a.pressure, b.pressure) and np.array_equal(a.u, b.u)
    finally:
        for g in grids:
            g.destroy()
