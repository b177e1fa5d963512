"""The operator and its triangular factors on many columns as matrix products."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


@pytest.mark.parametrize("n,wp", [(15, 1), (33, 2), (65, 8), (130, 9), (257, 17), (300, 40)])
def test_panel_products(n, wp):
    """The operator, L, L^-T, L^T and L^-1 on 2 to 80 columns as matrix products (tiles of 32 to 32 real
    columns, of 64 above), against the column-block kernel: an entry sums at most n products either way."""
    rng = np.random.default_rng(1000 * n + wp)
    _say(f"panel products n={n} wp={wp}")
    X = rng.normal(size=(n, n))
    S = X @ X.T / n + np.eye(n)
    h = (X + X.T) * 2.0
    bra = rng.normal(size=(wp, n)) + 1j * rng.normal(size=(wp, n))
    ket = rng.normal(size=(wp, n)) + 1j * rng.normal(size=(wp, n))
    res = {}
    with hip.Context(0) as ctx:
        for variant in (15, 9):
            hip.force_matvec_variant(variant)
            try:
                s = hip.System(ctx, n_orb=n, n_wp=wp, n_frag=1)
                s.load_operators(S, h)
                for w in range(wp):
                    s.set_wavepacket(w, S @ bra[w], ket[w])
                s.propagate(0.0, 1e-5)
                res[variant] = [np.stack([s.wavepacket(w)[i] for w in range(wp)]) for i in range(2)] + \
                               [np.stack([s.observables(w)[0] for w in range(wp)])] + \
                               [np.array([s.observables(w)[2] for w in range(wp)])]
                s.close()
            finally:
                hip.force_matvec_variant(-1)
    # condition of S is below 6 at these sizes; a few tens of products deep
    for a, b in zip(res[15], res[9]):
        assert np.abs(a - b).max() <= 200.0 * (n + 10) * np.finfo(np.float64).eps * np.abs(b).max()
