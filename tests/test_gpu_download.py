"""Fields read back whole, by every way a copy to the host takes."""
import ctypes

import numpy as np
import pytest

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
    from nextsimdg_amd.learned import DeviceArray

    print(f"download {nx}x{ny} {where}", flush=True)
    k = _kernel(nx, ny)
    want = np.random.default_rng(nx).normal(size=(nx * ny, 8))
    k.setData("s11", want, 8)

    def get(addr):
        check(k.lib.nsdg_dyn_get_field(k.h, b"s11", ctypes.cast(addr, ctypes.POINTER(ctypes.c_double)), 8))

    if where == "device":
        out = DeviceArray((want.size,), np.float64)
        get(out.ptr)
        assert np.array_equal(out.numpy(), want.ravel())
        return
    addr = ctypes.c_void_p()
    assert k.lib.hipHostMalloc(ctypes.byref(addr), ctypes.c_size_t(want.nbytes), 0) == 0
    try:
        out = np.ctypeslib.as_array(ctypes.cast(addr, ctypes.POINTER(ctypes.c_double)), (want.size,))
        out[:] = np.nan
        get(addr)
        assert np.array_equal(out, want.ravel())
    finally:
        k.lib.hipHostFree(addr)


def _round_trip(k, name, ncomp, scale):
    """A field of distinct values, set and read back into memory filled with NaN."""
    from nextsimdg_amd._lib import check, dptr

    want = scale * np.arange(1.0, k.ne * ncomp + 1.0)
    k.setData(name, want.reshape(k.ne, ncomp), ncomp)
    out = np.full(want.size, np.nan)
    check(k.lib.nsdg_dyn_get_field(k.h, name.encode(), dptr(out), ncomp))
    assert np.array_equal(out, want), (name, ncomp, np.flatnonzero(out != want)[:4])


# 3 * 2^18 values are 6 MiB, from where a copy is split: that size, two values less, a row
# more, odd sizes; with 8 components four threads, 513 x 515 two of 16 slots and a remainder.
@pytest.mark.parametrize("nx,ny", [(1024, 768), (393215, 2), (1024, 769), (1033, 1021), (513, 515), (397, 263)])
def test_fields_round_trip_around_the_split(nx, ny):
    print(f"round trip {nx}x{ny}", flush=True)
    k = _kernel(nx, ny)
    for ncomp in (1, 8):
        _round_trip(k, "s12", ncomp, 0.5)
    _round_trip(k, "hice", 6, 0.25)
    for n in ("u", "v"):
        want = np.arange(float(k.ncg)) - 7.0
        k.set_cg(n, want)
        assert np.array_equal(k.get_cg(n), want), n


def test_one_handle_small_large_small():
    """Two threads, four (new slots), two again, with other values each time; then plain copies."""
    k = _kernel(1061, 997)
    for i, (name, ncomp) in enumerate([("ssh", 1), ("s11", 1), ("s11", 8), ("s22", 1), ("hice", 6), ("s11", 1)]):
        _round_trip(k, name, ncomp, 1.0 + i)
    small = _kernel(31, 17)
    _round_trip(small, "s11", 8, 3.0)
