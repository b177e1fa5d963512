"""Where the device has no memory for the transfer buffer, matrices of other pitches go column by column."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [100, 700])
def test_without_the_transfer_buffer(N):
    print(f"[gpu] transfers by column, N={N}", flush=True)
    rng = np.random.default_rng(N)
    a, b, x = rng.normal(size=(3, N, N)) / (4.0 * N)
    S, h, X = np.eye(N) + a + a.T, -10.0 * np.eye(N) + b + b.T, x + x.T
    c = (rng.normal(size=(2, N)) + 1j * rng.normal(size=(2, N))) / np.sqrt(2.0 * N)
    out = []
    for forbid in (False, True):
        hip.forbid_transfer_buffer(forbid)
        try:
            with hip.Context(0) as ctx:
                s = hip.System(ctx, n_orb=N, n_wp=2)
                s.load_operators(S, h, want_hprime=True)
                for w in range(2):
                    s.set_initial_state(w, c[w], c[w])
                out.append([s.matrix(hip.DH_MAT_S), s.matrix(hip.DH_MAT_H), s.matrix(hip.DH_MAT_HPRIME),
                            s.ehrenfest_kernel(0, 1, X)])
                s.close()
        finally:
            hip.forbid_transfer_buffer(False)
    assert np.array_equal(out[1][0], S)
    for p, q in zip(*out):
        assert np.array_equal(p, q)
