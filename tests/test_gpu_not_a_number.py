"""An ocean velocity component that is not a number reaches both ice velocity components of
its node through the drag, as in IEEE arithmetic, and no other node within a subcycle."""
import numpy as np
import pytest

from helpers import box_coords


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["mevp", "mevp fp32", "mevp sphere", "bbm", "bbm warped"])
@pytest.mark.parametrize("component", ["uocean", "vocean"])
def test_nan_ocean_velocity_reaches_both_components(kind, component):
    print(f"{kind} {component}", flush=True)
    import nextsimdg_amd as nd
    from nextsimdg_amd import inputs

    nx, ny = 17, 15
    sph = "sphere" in kind
    coords = inputs.sphere_patch_coords(nx, ny, -0.2, 0.2, 0.9, 1.2) if sph else box_coords(nx, ny, 8000.0)
    if "warped" in kind:
        coords[:, 0] += 900.0 * np.sin(coords[:, 1] / 7000.0)
    k = (nd.BBMDynamicsKernel if "bbm" in kind else nd.MEVPDynamicsKernel)(2, 6)
    k.initialise(coords, sph, np.ones(nx * ny), nx, ny)
    one = np.ones(nx * ny)
    for n, v in (("hice", 1.0), ("cice", 0.9), ("uwind", 7.0), ("vwind", 4.0), ("uocean", 0.02), ("vocean", 0.01),
                 ("ssh", 0.0)):
        k.setData(n, v * one, 1)
    if "fp32" in kind:
        k.set_precision(1)
    k.prepareIteration()
    k.begin_iteration(120.0)
    node = (2 * nx + 1) * 12 + 9
    ocean = k.get_cg(component)
    ocean[node] = np.nan
    k.set_cg(component, ocean)
    k.subcycles(1)
    for n in ("u", "v"):
        assert np.array_equal(np.flatnonzero(np.isnan(k.get_cg(n))), [node]), n
