"""Atoms without orbitals (point charges, capping sites) are accepted and contribute nothing to S and h, however
many there are: far more than the operators have rows."""
import numpy as np
import pytest

from dynemol_amd import hip
from dynemol_amd.eht import Basis

pytestmark = pytest.mark.gpu


def _basis(shells):
    """shells[a]: number of s shells (n = 1, 2, ...) of atom a."""
    i4 = np.int32
    first = np.concatenate([[0], np.cumsum(shells)]).astype(i4)
    N = int(first[-1])
    n = np.concatenate([1 + np.arange(k) for k in shells]).astype(i4)
    zeta = np.zeros((N, 2))
    zeta[:, 0] = 1.0 + 0.07 * (np.arange(N) % 5)
    coef = np.tile([1.0, 0.0], (N, 1))
    zero = np.zeros(N, i4)
    atom = np.repeat(np.arange(len(shells)), shells).astype(i4)
    return Basis(len(shells), first, np.zeros(len(shells), i4), n, zero, zero, np.ones(N, i4), zeta, coef,
                 -10.0 - 0.1 * np.arange(N), np.full(N, 1.75), 0.01 * np.arange(N), atom, zero)


@pytest.mark.parametrize("with_orbitals,without", [(64, 136), (5, 400), (1, 200), (64, 0)])
def test_operators_of_the_atoms_with_orbitals(with_orbitals, without):
    """All atoms lie within the cutoff of each other; the ones with orbitals are spread among the others."""
    print(f"[gpu] {with_orbitals} atoms with and {without} without orbitals", flush=True)
    total = with_orbitals + without
    rng = np.random.default_rng(total)
    at = np.sort(rng.permutation(total)[:with_orbitals])
    shells = np.zeros(total, dtype=int)
    shells[at] = 1
    grid = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 3)[:total]
    coords = 0.8 * grid + rng.normal(0.0, 0.05, (total, 3))
    out = []
    with hip.Context(0) as ctx:
        for sh, x in ((shells, coords), (shells[at], coords[at])):
            s = hip.System(ctx, _basis(sh), n_wp=1, n_frag=1)
            s.set_coords(x)
            try:
                s.build()
            except hip.DHError:
                pass  # S need not be positive definite; S and h are there
            out.append((s.matrix(hip.DH_MAT_S), s.matrix(hip.DH_MAT_H)))
            s.close()
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    assert np.isfinite(out[0][0]).all()
