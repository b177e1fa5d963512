"""Outputs of all steps of a multi-step series in one product per operator, against one step at a time."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu

DT = 5.0e-4


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


@pytest.mark.parametrize("N,n_wp,steps", [(5, 1, 2), (33, 3, 7), (65, 1, 10), (130, 2, 23), (300, 12, 5), (500, 8, 10),
                                          (1025, 2, 9), (1500, 16, 4)])
def test_outputs_of_all_steps(N, n_wp, steps):
    """Populations, energies and the state read back.  The states of both runs agree to rounding of the series
    (1e-12 of the norm at these lengths), and so do bilinear sums of unit vectors."""
    _say(f"outputs N={N} n_wp={n_wp} steps={steps}")
    rng = np.random.default_rng(N)
    a, b = rng.normal(size=(2, N, N)) / np.sqrt(N)
    S, h = np.eye(N) + 0.1 * (a + a.T) / 2.0, 6.0 * (b + b.T) - 10.0 * np.eye(N)
    C = (rng.normal(size=(n_wp, N)) + 1j * rng.normal(size=(n_wp, N))) / np.sqrt(2.0 * N)
    res = []
    with hip.Context(0) as ctx:
        for per_series in (0, 1):
            s = hip.System(ctx, n_orb=N, n_wp=n_wp, n_frag=1)
            s.load_operators(S, h)
            s.set_steps_per_series(per_series)
            for w in range(n_wp):
                s.set_initial_state(w, C[w], C[w])
            pops, erg, _ = s.propagate_steps(steps, DT)
            state = [np.stack([x[i] for x in (s.wavepacket(w) for w in range(n_wp))]) for i in range(2)]
            obs = [s.observables(w) for w in range(n_wp)]
            res.append([pops, erg, *state, np.stack([o[0] for o in obs]), np.stack([o[1] for o in obs]),
                        np.array([o[2] for o in obs])])
            s.close()
    for x, y in zip(*res):
        assert np.abs(x - y).max() <= 1e-11 * np.abs(y).max()
    # the last step's observables are the ones read afterwards
    assert np.array_equal(res[0][0][-1], res[0][5])
    assert np.array_equal(res[0][1][-1], res[0][6])
