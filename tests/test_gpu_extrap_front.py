"""The extrapolation's front on the GPU where its bookkeeping can go wrong:
pass ceilings from one to the most, fronts that die out early, bands of a few
cells and of more than a workgroup, cells whose six neighbours leave the grid,
rows that no vector load divides, and two surfaces in turn on one grid.  Bar:
bit for bit against the CPU restatement, the report's counts included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def surface(dims, seed, kind):
    rng = np.random.default_rng(seed)
    c = [np.arange(n) / max(dims) for n in dims]
    x, y, z = np.meshgrid(*c, indexing="ij")
    if kind == "specks":  # a few wet cells
        phi = np.ones(dims)
        for _ in range(3):
            phi[tuple(rng.integers(0, n) for n in dims)] = -1.0
    elif kind == "rough":
        phi = y - 0.4 * dims[1] / max(dims) + 0.2 * np.sin(8 * x + seed) * np.cos(6 * z) + 0.05 * rng.standard_normal(dims)
    else:  # nearly full: the front has nowhere to go
        phi = np.where(rng.uniform(size=dims) < 0.02, 1.0, -1.0)
    vel = [rng.standard_normal((dims[0] + (a == 0), dims[1] + (a == 1), dims[2] + (a == 2))).astype(np.float32)
           for a in range(3)]
    return phi.astype(np.float32), vel, 1.0 / max(dims)


@pytest.mark.parametrize("dims", [(5, 7, 3), (16, 16, 16), (33, 18, 21), (12, 40, 67), (2, 9, 130)])
@pytest.mark.parametrize("open_top", [False, True])
def test_front_bit_exact(fpl, oracle, dims, open_top):
    g = None
    try:
        for seed, (kind, passes) in enumerate((("specks", 0), ("rough", 1), ("rough", 2), ("full", 0), ("rough", 16),
                                               ("rough", 0))):
            phi, vel, h = surface(dims, seed, kind)
            g = g or fpl.UniformPressureProjection(dims, h)
            for field in ("phi", "density"):
                f = phi if field == "phi" else np.clip(0.5 - phi, 0, 1).astype(np.float32)
                want = oracle.extrapolate(*vel, h, open_top=int(open_top), max_passes=passes, **{field: f})
                got = g.extrapolate(*vel, open_top=open_top, max_passes=passes, **{field: f})
                for a, b in zip(got[:3], want[:3]):
                    assert np.array_equal(a, b), (kind, passes, field)
                rep, orep = got[3], want[3]
                assert (rep["passes"], rep["active_left"]) == (orep["passes"], orep["active_left"]), (kind, passes)
                assert (rep["band_faces"], rep["unknown_faces"]) == (orep["band_known"], orep["unknown"])
    finally:
        if g:
            g.destroy()


# the first coarse level above the size that takes tiles, odd itself and no multiple of a tile on any axis
@pytest.mark.parametrize("dims", [(205, 213, 209)])
def test_tiled_levels_bit_exact(fpl, oracle, dims):
    phi, vel, h = surface(dims, 3, "rough")
    g = fpl.UniformPressureProjection(dims, h)
    try:
        want = oracle.extrapolate(*vel, h, phi=phi)
        got = g.extrapolate(*vel, phi=phi)
        for a, b in zip(got[:3], want[:3]):
            assert np.array_equal(a, b)
    finally:
        g.destroy()
