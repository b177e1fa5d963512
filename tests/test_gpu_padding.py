"""Only off its diagonal does the padding of a caller's operator have to be zero: what stands on the diagonal of rows
past N does not matter, and does not cost a repeat by other kernels (the same bits as with zeros there)."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu
DT = 5.0e-4


@pytest.mark.parametrize("N,R", [(130, 1), (500, 4), (1100, 8), (2500, 8), (3000, 4), (4030, 2)])
def test_padded_diagonal(N, R):
    print(f"[gpu] padded diagonal, N={N}, R={R}", flush=True)
    ld = (N + 63) // 64 * 64
    rng = np.random.default_rng(N)
    x = rng.normal(size=(N, N))
    H = np.zeros((ld, ld))
    H[:N, :N] = (x + x.T) * (34.0 / np.sqrt(8.0 * N))
    phi = np.zeros((ld, R), dtype=complex)
    phi[:N] = (rng.normal(size=(N, R)) + 1j * rng.normal(size=(N, R))) / np.sqrt(2.0 * N)
    out = []
    with hip.Context(0) as ctx:
        bufs = [hip.DeviceBuffer(n) for n in (H.nbytes, phi.nbytes, hip.chebyshev_work_bytes(N, R))]
        for pad in (0.0, 1e300, np.inf, np.nan):
            H[np.arange(N, ld), np.arange(N, ld)] = pad
            bufs[0].upload(H)
            bufs[1].upload(phi)
            hip.chebyshev_apply(ctx, N, bufs[0].ptr, ld, [-36.0, 36.0], DT, R, bufs[1].ptr, bufs[2].ptr, bufs[2].nbytes)
            out.append(bufs[1].download((ld, R), np.complex128))
        for b in bufs:
            b.close()
    for o in out:
        assert np.array_equal(o, out[0])
        assert not o[N:].any()
