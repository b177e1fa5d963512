"""Host matrices of other pitches than the device's: loaded and read back bit for bit."""
import ctypes

import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu
D = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


# N = 64: the device's pitch; 100 (device pitch 128) with the host's own, the device's, and wider pitches (past
# 2 N one column at a time); 2100: several blocks of columns
@pytest.mark.parametrize("N,ld", [(1, 1), (64, 64), (64, 70), (100, 100), (100, 128), (100, 150), (100, 201),
                                  (2100, 2100), (2100, 2150)])
def test_load_and_read_back(ctx, N, ld):
    rng = np.random.default_rng(N + ld)
    S = np.full((ld, N), np.nan, order="F")  # the caller's padding rows must stay out
    h = np.full((ld, N), np.nan, order="F")
    a, b = rng.normal(size=(2, N, N)) / (4.0 * N)
    S[:N] = np.eye(N) + a + a.T
    h[:N] = -10.0 * np.eye(N) + b + b.T
    print(f"[gpu] matrices of pitch {ld}, N={N}", flush=True)
    s = hip.System(ctx, n_orb=N, n_wp=1)
    L = hip.lib()
    assert L.dh_load_operators(s.h, S.ctypes.data_as(D), h.ctypes.data_as(D), ld) == 0
    assert L.dh_orthogonalize(s.h, 0) == 0
    for which, ref in ((hip.DH_MAT_S, S), (hip.DH_MAT_H, h)):
        assert np.array_equal(s.matrix(which), ref[:N])
        out = np.full((ld, N), 3.0, order="F")
        assert L.dh_get_matrix(s.h, which, out.ctypes.data_as(D), ld) == 0
        assert np.array_equal(out[:N], ref[:N])
        if ld != (N + 63) // 64 * 64:
            assert np.all(out[N:] == 3.0)
    assert np.isfinite(s.matrix(hip.DH_MAT_HORTH)).all()
    s.close()
