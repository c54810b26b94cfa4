"""Large downloads into memory that is not ordinary host memory: pinned, and on
the device (hipMemcpy takes both).  The bytes that were uploaded."""
import ctypes as C

import numpy as np
import pytest

from combustioncodegpu_amd import abi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("device", [False, True])
def test_download_into(device):
    from combustioncodegpu_amd.lib import Solver
    case = cases.c1(131, 77, 88, n_spec=9)  # cv: 107 MiB
    g = Solver(case)
    shp = case.blocks[0].padded_shape
    rng = np.random.default_rng(1)
    cv, bv, yk = (rng.standard_normal((n,) + shp) for n in (14, 6, 9))
    g.upload_state(0, cv, bv, yk)
    print(f"[copy] {cv.nbytes / 2**20:.1f} MiB into {'device' if device else 'pinned'} memory", flush=True)
    hip = g.lib  # the runtime that the library is linked with
    dst, n = C.c_void_p(), C.c_size_t(cv.nbytes)
    assert (hip.hipMalloc(C.byref(dst), n) if device else hip.hipHostMalloc(C.byref(dst), n, C.c_uint(0))) == 0
    got = np.zeros_like(cv)
    for _ in range(2):
        assert g.lib.cfx_download(g.h, 0, abi.CV, C.cast(dst, C.POINTER(C.c_double))) == 0
        assert hip.hipDeviceSynchronize() == 0
        got[:] = 0.0
        assert hip.hipMemcpy(C.c_void_p(got.ctypes.data), dst, n, 4) == 0  # hipMemcpyDefault
        assert np.array_equal(got, cv)
    assert np.array_equal(g.download(0, abi.CV), cv)
    assert (hip.hipFree(dst) if device else hip.hipHostFree(dst)) == 0
    g.close()
