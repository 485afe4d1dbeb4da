"""The advection's sample paths on the GPU: cells at every wall and edge of
grids down to two cells, rows that end inside a wave, flows of a fraction of a
cell and of several pieces, no flow, tiny and huge values, and quotients by h
either side of where the division takes over.  Bar: bit for bit against
the CPU restatement, both schemes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (2, 5, 66), (3, 2, 130), (17, 9, 2), (12, 20, 64), (21, 18, 33)])
@pytest.mark.parametrize("scheme", ["semi-lagrangian", "maccormack"])
def test_paths_bit_exact(fpl, oracle, dims, scheme):
    rng = np.random.default_rng(sum(dims))
    h = 1.0 / max(dims)
    y = np.arange(dims[1]) + 0.5
    phi = np.broadcast_to((y - 0.6 * dims[1])[None, :, None] * h, dims).astype(np.float32).copy()
    shapes = [(dims[0] + (a == 0), dims[1] + (a == 1), dims[2] + (a == 2)) for a in range(3)]
    g = fpl.UniformPressureProjection(dims, h)
    try:
        for cells, top in ((0.3, False), (0.3, True), (2.7, False), (9.0, True), (0.0, False), (1e-30, True),
                           (1e30, False), (None, True)):
            dt = 0.01
            field = [(rng.standard_normal(s) * cells * h / dt if cells is not None else
                      rng.uniform(-1.2e38, 1.2e38, s) * h).astype(np.float32) for s in shapes]
            cur = [(rng.standard_normal(s)).astype(np.float32) for s in shapes]
            want = oracle.advect_velocity(*cur, h, dt, phi=phi, transport=field, gravity=-9.81, nu=1e-3, scheme=scheme,
                                          open_top=int(top))
            got = g.advect(*cur, dt, phi=phi, transport=field, gravity=-9.81, viscosity=1e-3, scheme=scheme,
                           open_top=top)
            for a, b in zip(got[:3], want):
                assert np.array_equal(a, b, equal_nan=True), (cells, top)
    finally:
        g.destroy()


@pytest.mark.parametrize("h", [3e-36, 7e-34, 2e-31, 5e-29, 3e-27, 1e-24, 1e-20])
def test_tiny_cells(fpl, oracle, h):
    """Cell sizes at which a residual of the quotient by h, 2^-48 of the dividend, is subnormal."""
    dims = (9, 12, 33)
    rng = np.random.default_rng(4)
    phi = np.full(dims, -h, np.float32)
    shapes = [(dims[0] + (a == 0), dims[1] + (a == 1), dims[2] + (a == 2)) for a in range(3)]
    field = [(rng.standard_normal(s) * 0.7 * h).astype(np.float32) for s in shapes]
    cur = [rng.standard_normal(s).astype(np.float32) for s in shapes]
    g = fpl.UniformPressureProjection(dims, h)
    try:
        want = oracle.advect_velocity(*cur, h, 1.0, phi=phi, transport=field, gravity=0.0, nu=0.0,
                                      scheme="semi-lagrangian", open_top=0)
        got = g.advect(*cur, 1.0, phi=phi, transport=field, gravity=0.0, viscosity=0.0, scheme="semi-lagrangian",
                       open_top=False)
        for a, b in zip(got[:3], want):
            assert np.array_equal(a, b, equal_nan=True)
    finally:
        g.destroy()


@pytest.mark.parametrize("dims", [(3, 2, 130), (12, 20, 64), (21, 18, 33)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_non_finite_transport(fpl, oracle, dims, value):
    """A wave that meets a face that is not finite samples its first stage in
    full (0 times an infinity is not 0).  Its faces out of reach of that one,
    more than three cells away in a flow of a third of a cell, keep the bits of
    the finite field.  (What a face in reach becomes is not compared: clamps
    of a NaN differ between the device and C.)"""
    rng = np.random.default_rng(sum(dims))
    h, dt = 1.0 / max(dims), 0.01
    y = np.arange(dims[1]) + 0.5
    phi = np.broadcast_to((y - 0.6 * dims[1])[None, :, None] * h, dims).astype(np.float32).copy()
    shapes = [(dims[0] + (a == 0), dims[1] + (a == 1), dims[2] + (a == 2)) for a in range(3)]
    field = [(rng.uniform(-0.33, 0.33, s) * h / dt).astype(np.float32) for s in shapes]
    cur = [rng.standard_normal(s).astype(np.float32) for s in shapes]
    options = dict(phi=phi, gravity=-9.81, scheme="semi-lagrangian")
    want = oracle.advect_velocity(*cur, h, dt, transport=field, nu=0.0, open_top=0, **options)
    g = fpl.UniformPressureProjection(dims, h)
    try:
        for c in range(3):
            at = tuple(int(rng.integers(0, n)) for n in shapes[c])
            broken = [f.copy() for f in field]
            broken[c][at] = value
            got = g.advect(*cur, dt, transport=broken, viscosity=0.0, open_top=False, **options)
            for a, b in zip(got[:3], want):
                d = np.max([np.abs(np.arange(n) - q).reshape([-1 if k == j else 1 for j in range(3)]) * np.ones(a.shape)
                            for k, (n, q) in enumerate(zip(a.shape, at))], axis=0)
                assert np.array_equal(a[d > 3], b[d > 3]), (c, at)
            assert not all(np.array_equal(a, b) for a, b in zip(got[:3], want)), (c, at)
    finally:
        g.destroy()
