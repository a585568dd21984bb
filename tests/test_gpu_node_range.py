"""A mesh with more than 2^28 CG nodes, whose 16-byte node entries lie past byte 2^32."""
import numpy as np
import pytest

from helpers import box_coords, rel_l2


@pytest.mark.gpu
def test_nodes_past_the_first_2_to_28():
    """Three subcycles (a pair and a single pass) on a 16 x 4067300 mesh against three single
    passes, whose loads are indexed in 64 bits, on its nodes from 2^28 on. FP64: an ulp per
    operation, the bound of the other comparisons of passes. FP32: the random bits of the
    rounding go by a running count; a stress rounding is 6e-8 of the stress and less of the
    velocity, 1e-5 (another node's coefficients are wrong by a part in ten)."""
    import nextsimdg_amd as nd

    nx, ny, past = 16, 4067300, 2**28
    k = nd.MEVPDynamicsKernel(2, 6)
    k.initialise(box_coords(nx, ny, 4096.0), False, np.ones(nx * ny), nx, ny)
    print(f"{k.ncg} CG nodes", flush=True)
    assert k.ncg > past + 100 * (2 * nx + 1)
    j = np.arange(ny, dtype=np.float64)
    for name, v in (("hice", 1.0 + 0.1 * np.cos(0.4 * j)), ("cice", 0.9 + 0.05 * np.sin(0.3 * j)),
                    ("uwind", 8.0 + 2.0 * np.sin(0.7 * j)), ("vwind", 5.0 * np.cos(0.9 * j)),
                    ("uocean", 0.02 * np.sin(0.5 * j)), ("vocean", 0.01 * np.cos(0.6 * j)), ("ssh", 0.0 * j)):
        k.setData(name, np.repeat(v, nx), 1)
    k.prepareIteration()
    k.begin_iteration(120.0)
    zero, none = np.zeros(k.ncg), np.zeros(nx * ny)
    for precision, tol in ((0, 1e-12), (1, 1e-5)):
        k.set_precision(precision)
        out = []
        for pairing in (1, 2):
            for n in ("u", "v"):
                k.set_cg(n, zero)
            for n in ("s11", "s12", "s22"):
                k.setData(n, none, 1)
            k.set_pairing(pairing)
            k.subcycles(3)
            out.append([k.get_cg(n)[past:] for n in ("u", "v")])
        for got, want in zip(*out):
            assert np.abs(want).max() > 0
            assert rel_l2(got, want) < tol, (precision, rel_l2(got, want))
