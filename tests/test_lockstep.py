"""The operators' kernels on the CPU stand-in (tests/cpp/lockstep), whose waves progress as unevenly as the
barriers allow: what a missing barrier would only rarely show on the card fails here every time."""
import ctypes

import numpy as np
import pytest

import lockstep_lib as L
import oracle_lib as O
from ahead_amd import an, datagen

pytestmark = pytest.mark.skipif(not L.available(), reason="no clang++ of ROCm to compile the kernels for the CPU")


@pytest.fixture(params=[0, 1], ids=["ascending", "descending"])
def waves(request):
    lib = L.lib()
    lib.lockstep_set(request.param, 0, 1)
    yield request.param
    lib.lockstep_set(0, 0, 4)


@pytest.mark.parametrize("n,bad", [(5, 1), (16 * 1024 * 2 + 77, 3)])
def test_single_pass_engine_under_uneven_waves(waves, n, bad):
    """A workgroup's waves agree on every tile they take, the first one included."""
    rng = np.random.default_rng(n)
    meta = an.an_meta(an.RESINT, 65117)
    codes = datagen.encode(rng.integers(0, 1 << 32, n).astype(np.uint64), meta.a, 8)
    codes[rng.choice(n, bad, replace=False)] ^= np.uint64(1 << 40)
    ref = O.check_and_decode_an(O.Col(codes, meta))
    dec, err, cnt = np.zeros(n, np.uint32), np.zeros(bad, np.uint64), np.full(2, 77, np.uint64)
    ws, col = L.Workspace(), L.column(codes, meta)
    for _ in range(2):
        L.check(L.lib().ahead_hip_check_and_decode_an(ctypes.byref(col), an.A_OID_ERR, dec.ctypes.data, n,
                                                      err.ctypes.data, bad, cnt.ctypes.data, ws.h, None))
        assert cnt.tolist() == [n - bad, bad]
        assert np.array_equal(dec[:n - bad], ref[0]) and np.array_equal(err, ref[1])
        cnt[:] = 77
