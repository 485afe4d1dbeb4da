"""fp_tall_remesh on columns that its closed forms have to get right: level
sets that change sign inside the tall cell (found by bisection), wet lids,
bases of 2, signed zeros, huge, infinite and NaN samples, and neighbour limits
that travel across whole lines of odd length.  Bar: bit for bit against the
row-by-row numpy restatement."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,ny,band,delta,odd", [(7, 5, 40, 8, 3, False), (70, 67, 96, 24, 4, False),
                                                     (3, 130, 64, 16, 1, False), (9, 64, 32, 24, 2, False),
                                                     (12, 10, 48, 12, 4, True)])
def test_columns(fpl, nx, nz, ny, band, delta, odd):
    import tall_remesh  # oracle/
    rng = np.random.default_rng(nx * nz + ny)
    h = 1.0 / ny
    # bases that fall and rise along the lines, limited; some columns at the least base
    raw = rng.integers(2, ny - band + 1, size=(nx, nz))
    raw[rng.uniform(size=raw.shape) < 0.1] = 2
    bases = tall_remesh.limit(raw, delta).astype(np.int32)
    P, S = band + 2, band + 2 + delta
    phi = rng.uniform(-5 * h, 5 * h, size=(nx, P, nz)).astype(np.float32)
    flip = rng.uniform(size=(nx, nz))
    phi[:, 0] = np.where(flip < 0.4, -np.abs(phi[:, 0]), np.abs(phi[:, 0]))   # many change sign inside the tall cell
    phi[:, 1] = np.where(flip < 0.2, np.abs(phi[:, 1]), phi[:, 1])
    phi[rng.uniform(size=phi.shape) < 0.02] = np.float32(-0.0)
    phi[rng.uniform(size=phi.shape) < 0.02] = np.float32(1e30)
    phi[rng.uniform(size=phi.shape) < 0.02] = np.float32(-1e-38)
    # some columns dry, some wet up to the band's top
    phi[:, :, nz // 2] = 5 * h
    phi[nx // 2] = -5 * h
    u = rng.standard_normal((nx + 1, S, nz)).astype(np.float32)
    v = rng.standard_normal((nx, P, nz)).astype(np.float32)
    w = rng.standard_normal((nx, S, nz + 1)).astype(np.float32)
    v[rng.uniform(size=v.shape) < 0.02] = np.float32(-0.0)
    if odd:
        phi[0, 0, 0], phi[1, 1, 1], phi[2, 0, 2], phi[3, 4, 3] = np.nan, np.inf, -np.inf, np.nan
        v[4, 0, 4], u[5, 0, 5], w[6, 1, 6] = np.inf, np.nan, -np.inf
    g = fpl.TallCellPressureProjection(bases, ny, band, h, delta)
    try:
        with np.errstate(all="ignore"):
            want = tall_remesh.remesh(bases, phi, u, v, w, ny, band, delta, h)
        got = g.remesh(phi, u, v, w)
        assert np.array_equal(g.bases, want[0])
        assert got[4] == want[5] and got[4] > 0
        for a, b in zip(got[:4], want[1:5]):
            assert np.array_equal(a, b, equal_nan=True)
            assert np.array_equal(np.signbit(a[~np.isnan(a)]), np.signbit(b[~np.isnan(b)]))
    finally:
        g.destroy()
