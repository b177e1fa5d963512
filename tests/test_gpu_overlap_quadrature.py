"""S and h of the device's quadrature against the oracle's closed forms, over the exponents, distances and
orientations at which its parts change: the point counts' edges in |t| = |za - zb| R / 2 (4, 16), the shortened
eta interval (|t| > 40), bonds along the axes, two exponents per shell, the cutoff, and pair counts that are no
multiple of a wave's.

The quadrature is good to rounding; the closed forms lose digits to cancellation at short bonds with nearly
equal exponents: against an independent 64-point quadrature up to 1.6e-12 (5000 random shell pairs of these
ranges), and below 7e-15 for |t| >= 4."""
import numpy as np
import pytest

from dynemol_amd import hip
from dynemol_amd.eht import Basis
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"[gpu] {msg}", flush=True)


def _basis(atoms):
    """atoms: per atom a list of shells (n, l, exponents, coefficients)."""
    rows, first, lmax = [], [0], []
    for ia, shells in enumerate(atoms):
        for n, l, z, c in shells:
            rows += [(n, l, m, len(z), (list(z) + [0.0])[:2], (list(c) + [0.0])[:2], ia) for m in range(-l, l + 1)]
        first.append(len(rows))
        lmax.append(max(s[1] for s in shells))
    N = len(rows)

    def col(k, t):
        return np.array([r[k] for r in rows], dtype=t)

    i4 = np.int32
    return Basis(len(atoms), np.array(first, i4), np.array(lmax, i4), col(0, i4), col(1, i4), col(2, i4), col(3, i4),
                 col(4, float).reshape(N, 2), col(5, float).reshape(N, 2), -10.0 - 0.1 * np.arange(N),
                 np.full(N, 1.75), 0.01 * np.arange(N), col(6, i4), np.zeros(N, i4))


def _compare(coords, atoms, tol, cutoff=12.0):
    b = _basis(atoms)
    coords = np.ascontiguousarray(coords, dtype=np.float64)
    S = O.overlap(coords, b, cutoff)
    h = O.huckel(b, S)
    with hip.Context(0) as ctx:
        s = hip.System(ctx, b, n_wp=1, n_frag=1)
        s.set_coords(coords)
        try:
            s.build(cutoff=cutoff)
        except hip.DHError:
            pass  # S of such a set need not be positive definite; S and h are there
        ds = np.abs(s.matrix(hip.DH_MAT_S) - S).max()
        dh = np.abs(s.matrix(hip.DH_MAT_H) - h).max()
        s.close()
    _say(f"  N={b.N} |dS|={ds:.1e} |dh|={dh:.1e}")
    assert ds <= tol
    assert dh <= 100.0 * tol  # |X| stays below 100 for these IPs


@pytest.mark.parametrize("za,zb,tol", [(1.3, 1.3, 1e-11), (1.0, 1.9, 1e-11), (0.7, 4.0, 1e-11), (1.0, 12.0, 1e-11)])
@pytest.mark.parametrize("axis", [(0, 0, 1), (1, 0, 0), (0, -1, 0), (1, 2, -3)])
def test_pairs_of_shells(za, zb, tol, axis):
    """Every pair of orders and principal quantum numbers up to 5, at distances through the tiers of |t|."""
    _say(f"pairs za={za} zb={zb} axis={axis}")
    u = np.array(axis, dtype=float) / np.linalg.norm(axis)
    for la in range(3):
        for lb in range(3):
            for na, nb in ((la + 1, 5), (4, lb + 1), (5, 5)):
                if abs(za - zb) * 5.5 >= 16.0 and la == lb == 2 and na == nb == 5:
                    r = 11.9  # |t| > 40 for the widest pair
                else:
                    r = (1.1, 2.9, 7.3)[(na + nb + la) % 3]
                _compare([[0.0, 0.0, 0.0], list(r * u)],
                         [[(na, la, [za], [1.0])], [(nb, lb, [zb], [1.0])]], tol)


@pytest.mark.parametrize("n_atoms,cutoff", [(2, 12.0), (9, 12.0), (24, 6.0)])
def test_many_atoms(n_atoms, cutoff):
    """Two-exponent d shells among s and p; some pairs beyond the cutoff; 1, 36 and up to 276 pairs of atoms."""
    _say(f"atoms {n_atoms} cutoff {cutoff}")
    rng = np.random.default_rng(n_atoms)
    grid = np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n_atoms]
    coords = 3.1 * grid + rng.normal(0.0, 0.2, (n_atoms, 3))
    atoms = []
    for i in range(n_atoms):
        shells = [(2 + i % 3, 0, [1.2 + 0.1 * (i % 4)], [1.0]), (2 + i % 3, 1, [1.1 + 0.2 * (i % 3)], [1.0])]
        if i % 2 == 0:
            shells.append((3, 2, [4.55, 1.4], [0.4206, 0.7839]))
        atoms.append(shells)
    _compare(coords, atoms, 1e-11, cutoff)
