"""The V-cycle's small levels on the GPU: the one-workgroup bottom in LDS
(against the FP64 oracle) and whole legs as one launch (against one launch per
sweep, residual and transfer, which a persistent projection takes: the same
bits)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def blob_case(dims, seed):
    """A level set with an uneven surface, bubbles and droplets, and a random right-hand side on liquid cells."""
    rng = np.random.default_rng(seed)
    c = [np.arange(n) / max(dims) for n in dims]
    x, y, z = np.meshgrid(*c, indexing="ij")
    phi = y - 0.55 * dims[1] / max(dims) + 0.15 * np.sin(9 * x + seed) * np.cos(7 * z) + 0.02 * rng.standard_normal(dims)
    phi = phi.astype(np.float32)
    r = np.where(phi < 0, rng.standard_normal(dims), 0).astype(np.float32)
    return phi, r, 1.0 / max(dims)


# bottoms whose first level is 8^3, 15^3, just under 4096 cells, flat, and one that only one axis coarsens
@pytest.mark.parametrize("dims", [(16, 16, 16), (15, 15, 15), (15, 16, 17), (4, 90, 11), (30, 30, 30), (6, 6, 113),
                                  (3, 5, 7)])
def test_bottom_matches_oracle(fpl, oracle, dims):
    phi, r, h = blob_case(dims, sum(dims))
    g = fpl.UniformPressureProjection(dims, h)
    try:
        for sweeps in (1, 2, 3):
            z = g.probe_vcycle(phi, r, precision="fp32", pre_sweeps=sweeps, post_sweeps=sweeps)
            oz = oracle.vcycle(phi, r.astype(np.float64), pre=sweeps, post=sweeps)
            # FP32 relaxations of an FP64 reference: the bound of the 64^3 V-cycle test
            assert np.linalg.norm(z - oz) < 2e-5 * np.linalg.norm(oz), sweeps
    finally:
        g.destroy()


# one tile, ragged tiles, axes that do not coarsen, an odd row length, and both sides of the size limits of the legs (FP32,
# then two-byte storage)
@pytest.mark.parametrize("dims", [(16, 16, 16), (4, 16, 64), (17, 19, 23), (33, 20, 18), (40, 24, 17), (5, 33, 32),
                                  (64, 10, 21), (80, 81, 80), (81, 81, 81), (101, 101, 102),
                                  (102, 101, 102)])
@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16"])
def test_leg_bits(fpl, dims, precision):
    phi, r, h = blob_case(dims, sum(dims))
    g = fpl.UniformPressureProjection(dims, h)
    try:
        for sweeps in (1, 2, 3):
            z = [g.probe_vcycle(phi, r, precision=precision, pre_sweeps=sweeps, post_sweeps=sweeps, persistent=p)
                 for p in (0, 1)]
            assert np.isfinite(z[0]).all() and np.abs(z[0]).max() > 0
            assert np.array_equal(z[0], z[1]), (sweeps, np.abs(z[0] - z[1]).max())
    finally:
        g.destroy()


# tanks whose waves lie in air alone, in liquid alone and across a wall, an edge of a row or the surface
@pytest.mark.parametrize("dims", [(16, 40, 64), (9, 30, 200), (20, 33, 17)])
@pytest.mark.parametrize("fill", [0.5, 0.97])
def test_flat_tank_matches_oracle(fpl, oracle, dims, fill):
    rng = np.random.default_rng(dims[2])
    h = 1.0 / max(dims)
    y = np.arange(dims[1]) + 0.5 - fill * dims[1]
    phi = np.broadcast_to((y * h)[None, :, None], dims).astype(np.float32).copy()
    phi[dims[0] // 2, 1:4, :] = 0.3 * h  # a bubble line through the liquid
    r = np.where(phi < 0, rng.standard_normal(dims), 0).astype(np.float32)
    g = fpl.UniformPressureProjection(dims, h)
    try:
        z = g.probe_vcycle(phi, r, precision="fp32", pre_sweeps=2, post_sweeps=2)
        oz = oracle.vcycle(phi, r.astype(np.float64), pre=2, post=2)
        # the bound of the 64^3 V-cycle test
        assert np.linalg.norm(z - oz) < 2e-5 * np.linalg.norm(oz)
    finally:
        g.destroy()
