"""dh_chebyshev_apply from the shortest to the longest series: the device's coefficient table against the host's,
and the state against the exact one of a diagonal operator."""
import numpy as np
import pytest

from dynemol_amd import hip
from oracle import oracle as O

pytestmark = pytest.mark.gpu

N, LO, HI = 64, -42.0, 30.0


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


@pytest.mark.parametrize("x", [1e-13, 1e-6, 1e-2, 0.9, 7.0, 40.0, 133.0, 512.0, 1700.0])
def test_terms_and_state(x):
    """x = r dt.  A term's error is at most about its index times eps, and the coefficients' squares sum to
    about 1: K^1.5 eps over the K terms."""
    _say(f"apply x={x}")
    dt = x / (0.5 * (HI - LO)) * O.H_BAR
    rng = np.random.default_rng(int(1e6 * x) % 2**31)
    e = np.sort(rng.uniform(LO + 0.5, HI - 0.5, N))
    phi = rng.normal(size=(N, 2)) + 1j * rng.normal(size=(N, 2))
    phi /= np.linalg.norm(phi, axis=0)
    wb = hip.chebyshev_work_bytes(N, 2)
    with hip.Context(0) as ctx:
        h, p, w = hip.DeviceBuffer(8 * N * N), hip.DeviceBuffer(16 * N * 2), hip.DeviceBuffer(wb)
        h.upload(np.asfortranarray(np.diag(e)))
        p.upload(np.ascontiguousarray(phi))
        k = hip.chebyshev_apply(ctx, N, h.ptr, N, [LO, HI], dt, 2, p.ptr, w.ptr, wb)
        out = p.download((N, 2), np.complex128)
        for b in (h, p, w):
            b.close()
    _, K = hip.bessel_coefficients(x, 0.0)
    assert k == K + 1
    ref = np.exp(-1j * e * dt / O.H_BAR)[:, None] * phi
    assert np.abs(out - ref).max() <= 4.0 * (K + 10) ** 1.5 * np.finfo(np.float64).eps
