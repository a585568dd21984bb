"""DGTransport.run (normal velocities once, limiters in the last stage of a step) against the
same steps taken one by one with the limiters as calls of their own."""
import numpy as np
import pytest

from helpers import box_coords, rel_l2


@pytest.mark.gpu
@pytest.mark.parametrize("dg", [1, 3, 6])
@pytest.mark.parametrize("scheme", ["rk1", "rk2", "rk3"])
@pytest.mark.parametrize("nx,ny,warp", [(2, 2, 0.0), (16, 16, 0.0), (17, 31, 0.2)])
def test_run_equals_steps_and_limiters(dg, scheme, nx, ny, warp):
    """Land cells, walls and values on both limits; one block of 256 elements and more. Both
    run the same cell arithmetic, which the compiler may contract differently in the limiter's
    own kernel: an ulp per step, times the few steps."""
    print(f"transport run dg={dg} {scheme} {nx}x{ny}", flush=True)
    import nextsimdg_amd as nd
    from nextsimdg_amd.dynamics import LimitMax, LimitMin

    coords = box_coords(nx, ny, 1000.0, 900.0)
    coords[:, 0] += 1000.0 * warp * np.sin(coords[:, 1] / 700.0)
    mask = np.ones(nx * ny)
    if nx > 2:
        mask[(ny // 2) * nx + nx // 2] = 0.0
    m = nd.ParametricMesh(nx, ny, coords)
    m.landmaskFromModelArray(mask)
    m.dirichletFromMask()
    for e in range(4):
        m.dirichletFromEdge(e)
    t = nd.DGTransport(m, dg)
    t.settimesteppingscheme(scheme)
    rng = np.random.default_rng(dg * 100 + nx)
    vx, vy = (rng.normal(0, 1, (nx * ny, dg)) * np.r_[1.0, [0.2] * (dg - 1)] for _ in range(2))
    t.set_velocity(vx, vy)
    phi = rng.uniform(-0.2, 1.2, (nx * ny, dg)) * np.r_[1.0, [0.3] * (dg - 1)]
    for hi, lo in ((True, True), (True, False), (False, True), (False, False)):
        got = t.run(20.0, phi, 5, hi, lo)
        ref = phi
        for _ in range(5):
            t.reinitnormalvelocity()
            ref = t.step(20.0, ref)
            if hi:
                ref = LimitMax(dg, ref, 1.0)
            if lo:
                ref = LimitMin(dg, ref, 0.0)
        assert rel_l2(got, ref) < 1e-13, (hi, lo)
