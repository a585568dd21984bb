"""Fields read back whole, by every way a copy to the host takes."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import box_coords

pytestmark = pytest.mark.gpu


def _kernel(nx, ny):
    import nextsimdg_amd as nd

    k = nd.MEVPDynamicsKernel(2, 6)
    k.initialise(box_coords(nx, ny, 4000.0), False, np.ones(nx * ny), nx, ny)
    return k


@pytest.mark.parametrize("where", ["pinned", "device"])
@pytest.mark.parametrize("nx,ny", [(16, 16), (515, 513)])
def test_download_into_memory_the_runtime_knows(where, nx, ny):
    """Page-locked host memory and device memory as the destination, small and large."""
    from nextsimdg_amd._lib import check

    print(f"download {nx}x{ny} {where}", flush=True)
    k = _kernel(nx, ny)
    want = np.random.default_rng(nx).normal(size=(nx * ny, 8))
    k.setData("s11", want, 8)
    out = torch.empty(want.size, dtype=torch.float64, **({"pin_memory": True} if where == "pinned" else {"device": "cuda"}))
    torch.cuda.synchronize()
    check(k.lib.nsdg_dyn_get_field(k.h, b"s11", ctypes.cast(out.data_ptr(), ctypes.POINTER(ctypes.c_double)), 8))
    assert np.array_equal(out.cpu().numpy(), want.ravel())
