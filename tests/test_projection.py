"""The projection of the general meshes' kernels: through the Gauss weights instead of the
inverse mass matrix. On the CPU the identity itself, on the GPU strongly distorted elements
and large spherical ones, against the split passes with their inverse-mass tables."""
import numpy as np
import pytest

from helpers import box_coords, rel_l2


def _basis(x, y):
    X, Y, t = x - 0.5, y - 0.5, 1.0 / 12.0
    return np.stack([np.ones_like(X), X, Y, X * X - t, Y * Y - t, X * Y, Y * (X * X - t), X * (Y * Y - t)])


@pytest.mark.parametrize("S,G", [(8, 3), (3, 2)])
def test_projection_through_the_gauss_weights(S, G):
    """M^-1 PSI W r = (coefficients of r - n / W (sum n r) / (sum n^2 / W)) for any positive
    weights W. Rounding of the dense inverse: cond(M) < 2e4 (basis norms 1 to 1/2160, weights
    within a factor 6) times 1e-16 and a few tens of operations, below 1e-10."""
    p, w = np.polynomial.legendre.leggauss(G)
    p, w = 0.5 * (p + 1), 0.5 * w
    x, y, w2 = np.tile(p, G), np.repeat(p, G), np.tile(w, G) * np.repeat(w, G)
    B = _basis(x, y)[:S]
    n1 = np.array([1.0, -2.0, 1.0]) if G == 3 else np.array([1.0, -1.0])
    n = np.repeat(n1, G) * np.tile(n1, G)
    assert np.abs(B @ n).max() < 1e-15
    L = B * w2 / (B * B * w2).sum(1, keepdims=True)
    rng = np.random.default_rng(G)
    for _ in range(200):
        W, r = w2 * rng.uniform(0.5, 3.0, G * G), rng.normal(size=G * G)
        dense = np.linalg.solve((B * W) @ B.T, B @ (W * r))
        fast = L @ (r - n / W * (n @ r) / (n * n / W).sum())
        assert np.abs(dense - fast).max() < 1e-10 * np.abs(dense).max()


def _distorted(nx, ny):
    """Element sides and angles changing by half an element from vertex to vertex."""
    c = box_coords(nx, ny, 3000.0, 2500.0, skew=0.4)
    i, j = np.meshgrid(np.arange(nx + 1), np.arange(ny + 1))
    c[:, 0] += 600.0 * np.sin(2.1 * j.ravel() + 0.7 * i.ravel())
    c[:, 1] += 500.0 * np.cos(1.7 * i.ravel() - 0.4 * j.ravel())
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("cg,dg", [(2, 6), (1, 3)])
@pytest.mark.parametrize("mesh,nx,ny", [("distorted", 33, 15), ("distorted", 2, 9), ("sphere", 12, 7), ("sphere", 31, 8)])
def test_geometry_kernels_on_extreme_elements(cg, dg, mesh, nx, ny):
    """mEVP subcycles from the geometry against the split passes, with land and stored strain.
    The sphere patch spans 25 to 85 degrees north: elements of up to 9 degrees, over which
    the metric weight changes several-fold. Bound 1e-12, as for the other general meshes."""
    print(f"geometry kernels cg={cg} {mesh} {nx}x{ny}", flush=True)
    import nextsimdg_amd as nd
    from nextsimdg_amd import inputs

    S = 8 if cg == 2 else 3
    sph = mesh == "sphere"
    coords = inputs.sphere_patch_coords(nx, ny, -0.8, 0.8, 0.43, 1.48) if sph else _distorted(nx, ny)
    mask = np.ones(nx * ny)
    mask[(ny // 2) * nx + nx // 2] = 0.0
    ne, ncg = nx * ny, (cg * nx + 1) * (cg * ny + 1)
    rng = np.random.default_rng(nx * 100 + ny + cg)
    state = {"hice": np.abs(rng.normal(1.0, 0.3, (ne, dg))) * np.r_[1.0, [0.05] * (dg - 1)],
             "cice": np.clip(rng.normal(0.9, 0.05, (ne, dg)), 0, 1) * np.r_[1.0, [0.02] * (dg - 1)]}
    for n in ("s11", "s12", "s22", "e11", "e12", "e22"):
        state[n] = rng.normal(0, 1e3 if n[0] == "s" else 1e-7, (ne, S))
    forcing = {n: rng.normal(0, sc, ne) for n, sc in (("uwind", 10), ("vwind", 10), ("uocean", 0.05),
                                                       ("vocean", 0.05), ("ssh", 0.1))}
    vel = {n: rng.normal(0, 0.1, ncg) for n in ("u", "v")}
    ks = [nd.MEVPDynamicsKernel(cg, dg) for _ in range(2)]
    for k in ks:
        k.initialise(coords, sph, mask, nx, ny)
        for n, v in state.items():
            k.setData(n, v, v.shape[1])
        for n, v in forcing.items():
            k.setData(n, v, 1)
        for n, v in vel.items():
            k.set_cg(n, v)
        k.prepareIteration()
        k.begin_iteration(120.0)
    a, b = ks
    a.subcycles(5)
    for _ in range(5):
        b.projectVelocityToStrain()
        b.stressUpdateHighOrder(1)
        b.stressDivergence()
        b.updateMomentum()
        b.applyBoundaries()
    a.synchronize()
    for n in ("u", "v"):
        assert np.isfinite(a.get_cg(n)).all()
        assert rel_l2(a.get_cg(n), b.get_cg(n)) < 1e-12, n
    for n in ("s11", "s12", "s22", "e11", "e12", "e22"):
        assert rel_l2(a.getDGData(n, S), b.getDGData(n, S)) < 1e-12, n
