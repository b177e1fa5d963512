"""Which systems' series run in one launch, and what the others do.

The exchange ring (four slots and the flags) goes into the system's scratch for partial sums, which is sized for the
term kernels: it does not fit at N <= 256 with 2 or 4 wavepackets and N <= 512 with 3.  Those systems run term by
term, as one captured graph per step up to N = 2048."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu
DT = 5.0e-4


@pytest.mark.parametrize("N,n_wp,one_launch", [(1, 1, True), (60, 1, True), (256, 1, True), (200, 2, False),
                                               (256, 2, False), (257, 2, True), (256, 4, False), (257, 4, True),
                                               (512, 3, False), (513, 3, True), (4096, 2, True), (4097, 1, False),
                                               (3840, 4, True), (3841, 4, False), (400, 5, False)])
def test_form(N, n_wp, one_launch):
    print(f"[gpu] form of the series, N={N}, n_wp={n_wp}", flush=True)
    rng = np.random.default_rng(N)
    b = rng.normal(size=(N, N)) * (8.0 / np.sqrt(N))
    with hip.Context(0) as ctx:
        s = hip.System(ctx, n_orb=N, n_wp=n_wp)
        s.load_operators(np.eye(N), b + b.T)
        c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
        for w in range(n_wp):
            s.set_initial_state(w, c, c)
        s.propagate(0.0, DT)
        got, graphs = hip.series_form(s)
        s.propagate_steps(2, DT)
        several, _ = hip.series_form(s)
        retries = s.stats()["retries"]
        s.close()
    assert got == several == one_launch
    assert graphs == (0 if one_launch or N > 2048 else 1)
    assert retries == 0
