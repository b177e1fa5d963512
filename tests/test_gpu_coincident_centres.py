"""s shells on two centres at one point, or a tiny distance apart: S from the closed one-centre form.

int r^(n + n') e^(-(z + z') r) dr of the two normalised radial functions is
(2z)^(n + 1/2) (2z')^(n' + 1/2) (n + n')! / (sqrt((2n)! (2n')!) (z + z')^(n + n' + 1)), and the first
correction is of order (z R)^2, below 1e-19 at the distances here.  The quadrature's weights carry 16
digits and the powers about (n + n') roundings each: 1e-13 relative."""
import math

import numpy as np
import pytest

from dynemol_amd import hip
from dynemol_amd.eht import Basis

pytestmark = pytest.mark.gpu
i4 = np.int32


def _one_centre(n, z, m, y):
    f = math.factorial
    return ((2 * z) ** (n + 0.5) * (2 * y) ** (m + 0.5) * f(n + m)
            / (math.sqrt(f(2 * n) * f(2 * m)) * (z + y) ** (n + m + 1)))


@pytest.mark.parametrize("r", [0.0, 1e-30, 1e-14, 1e-10])
def test_s_shells_on_one_point(r):
    n = np.array([1, 2, 3, 5, 5], i4)
    z = np.array([1.3, 0.9, 2.1, 0.6, 4.5])
    print(f"[gpu] five s shells within {r}", flush=True)
    N = len(n)
    zero = np.zeros(N, i4)
    b = Basis(N, np.arange(N + 1, dtype=i4), zero, n, zero, zero, np.ones(N, i4), np.stack([z, 0 * z], 1),
              np.tile([1.0, 0.0], (N, 1)), np.full(N, -10.0), np.full(N, 1.75), np.zeros(N), np.arange(N, dtype=i4), zero)
    coords = np.full((N, 3), 0.7)
    coords[:, 2] = r * np.arange(N)
    coords[:, :2] *= 0.0 if r else 1.0
    with hip.Context(0) as ctx:
        s = hip.System(ctx, b, n_wp=1, n_frag=1)
        s.build(coords)
        S, H = s.matrix(hip.DH_MAT_S), s.matrix(hip.DH_MAT_HORTH)
        s.close()
    ref = np.array([[_one_centre(n[i], z[i], n[j], z[j]) for j in range(N)] for i in range(N)])
    assert np.abs(S / ref - 1.0).max() <= 1e-13
    assert np.isfinite(H).all()
