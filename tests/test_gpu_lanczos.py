"""The Lanczos recurrence in one launch against the one run step by step."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


@pytest.mark.parametrize("n", [64, 65, 130, 500, 513, 1025, 1537, 2049, 2561, 3073, 3585, 4096])
def test_lanczos_one_launch(n):
    """Sizes at the edges of a thread's share of columns.  The extreme Ritz values are backward stable: two
    orders of summation may differ by a few (n + steps) eps of the norm each step."""
    _say(f"lanczos n={n}")
    rng = np.random.default_rng(n)
    h = rng.normal(size=(n, n))
    h = (h + h.T) * (10.0 / np.sqrt(2.0 * n)) - 6.0 * np.eye(n)
    S = np.eye(n)
    out = {}
    with hip.Context(0) as ctx:
        for variant in (-1, 9):  # a forced kernel runs step by step
            hip.force_matvec_variant(variant)
            try:
                s = hip.System(ctx, n_orb=n, n_wp=1, n_frag=1)
                s.load_operators(S, h)
                out[variant] = s.bounds()
                s.close()
            finally:
                hip.force_matvec_variant(-1)
    a, b = out[-1], out[9]
    steps = min(48, n)
    tol = 4.0 * steps * (n + steps) * np.finfo(np.float64).eps * 30.0  # norm below 30
    assert np.abs(a[2:4] - b[2:4]).max() <= tol
    if n <= 1100:
        w = np.linalg.eigvalsh(h)
        assert a[0] <= w[0] and w[-1] <= a[1]
        assert a[2] >= w[0] - tol and a[3] <= w[-1] + tol
