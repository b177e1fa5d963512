"""A Chebyshev series in one launch with the operator resident on the chip (series.hip).

The same propagation term by term (a forced matvec variant) is the comparison:
both evaluate the same FP64 series of about 63 terms on an operator of half
width 34 eV, and the recurrence carries each term's rounding (a dot product of
N terms, below 1e-15 of the state's norm) at most K times, so the two differ by
less than 63^2 * 1e-15 = 4e-12 of the norm; 1e-11 is asserted.
"""
import numpy as np
import pytest

from dynemol_amd import hip
from dynemol_amd.structures import ch_cluster

pytestmark = pytest.mark.gpu
DT = 5.0e-4


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def operator():
    """One 4160 x 4160 symmetric matrix; its leading blocks are the operators."""
    rng = np.random.default_rng(5)
    x = rng.normal(size=(4160, 4160))
    return x + x.T


def _apply(ctx, operator, N, R, variant):
    ld = (N + 63) // 64 * 64
    H = np.eye(ld)
    H[:N, :N] = operator[:N, :N] * (34.0 / np.sqrt(8.0 * N))
    H[np.arange(N), np.arange(N)] -= 6.0
    rng = np.random.default_rng(N + R)
    phi = np.full((ld, R), 7.0 + 3.0j)  # rows past N: the call clears them
    phi[:N] = (rng.normal(size=(N, R)) + 1j * rng.normal(size=(N, R))) / np.sqrt(2.0 * N)
    bufs = [hip.DeviceBuffer(H.nbytes), hip.DeviceBuffer(phi.nbytes), hip.DeviceBuffer(hip.chebyshev_work_bytes(N, R))]
    try:
        bufs[0].upload(H)
        bufs[1].upload(phi)
        # a dirty work buffer: nothing in it may be taken for data
        bufs[2].upload(np.full(bufs[2].nbytes // 8, np.nan))
        hip.force_matvec_variant(variant)
        k = hip.chebyshev_apply(ctx, N, bufs[0].ptr, ld, [-42.0, 30.0], DT, R, bufs[1].ptr, bufs[2].ptr,
                                bufs[2].nbytes)
        return bufs[1].download((ld, R), np.complex128), k
    finally:
        hip.force_matvec_variant(-1)
        for b in bufs:
            b.close()


# edges of the tiles (16 rows and 128 columns per group of the 8 waves), of the register and LDS parts of
# the operator (N = 2944: the last of it in registers at R = 4), of the rows per workgroup at R = 8
# (2048) and of the sizes that stay resident (3584 at R = 8, 4096); 3585 and 4097 run term by term
@pytest.mark.parametrize("N,R", [(1, 2), (16, 4), (63, 1), (64, 8), (65, 4), (129, 2), (130, 8), (960, 4), (1025, 8),
                                 (1100, 4), (2048, 8), (2049, 8), (2944, 4), (3000, 4), (3009, 1), (3584, 8),
                                 (3585, 8), (4096, 4), (4096, 2), (4097, 2)])
def test_series_matches_terms(ctx, operator, N, R):
    print(f"[gpu] series in one launch, N={N}, R={R}", flush=True)
    a, ka = _apply(ctx, operator, N, R, -1)
    b, kb = _apply(ctx, operator, N, R, 1)
    assert ka == kb
    assert np.linalg.norm(a - b) <= 1e-11 * np.linalg.norm(b)
    assert np.abs(a[N:]).max(initial=0.0) == 0.0


@pytest.mark.parametrize("variant", [15, 18, -1])
def test_short_series_after_a_long_one(ctx, variant):
    """The coefficient rows of a longer series do not leak into the next one's accumulators."""
    st = ch_cluster(seed=1)
    b = st.basis()
    c = np.random.default_rng(3).normal(size=b.N) / np.sqrt(b.N) + 0j
    hip.force_matvec_variant(variant)
    try:
        out = []
        for before in (0.0, 4 * DT):
            s = hip.System(ctx, b, n_wp=1, n_frag=2)
            s.build(st.coords)
            if before:
                s.set_initial_state(0, c, c)
                s.propagate_steps(10, before)
            s.set_initial_state(0, c, c)
            s.set_steps_per_series(0 if before else 1)
            out.append(s.propagate_steps(10, DT)[0])
            s.close()
    finally:
        hip.force_matvec_variant(-1)
    assert np.abs(out[0] - out[1]).max() < 1e-12 * np.abs(out[0]).max()


@pytest.mark.parametrize("n_wp,n_steps", [(1, 1), (2, 23), (3, 12), (4, 11)])
def test_multi_step_series(ctx, n_wp, n_steps):
    """Several accumulators per series (up to 10 steps), 2 to 8 columns."""
    st = ch_cluster(seed=1)
    b = st.basis()
    rng = np.random.default_rng(n_wp)
    c = (rng.normal(size=(n_wp, b.N)) + 1j * rng.normal(size=(n_wp, b.N))) / np.sqrt(2.0 * b.N)
    out = []
    for variant in (-1, 1):
        hip.force_matvec_variant(variant)
        try:
            s = hip.System(ctx, b, n_wp=n_wp, n_frag=2)
            s.build(st.coords)
            for w in range(n_wp):
                s.set_initial_state(w, c[w], c[w])
            pops, erg, _ = s.propagate_steps(n_steps, DT)
            out.append((pops, erg, np.stack([s.wavepacket(w)[1] for w in range(n_wp)])))
            s.close()
        finally:
            hip.force_matvec_variant(-1)
    assert np.abs(out[0][0] - out[1][0]).max() < 1e-11 * np.abs(out[1][0]).max()
    assert np.abs(out[0][1] - out[1][1]).max() < 1e-11 * np.abs(out[1][1]).max()
    assert np.linalg.norm(out[0][2] - out[1][2]) <= 1e-11 * np.linalg.norm(out[1][2])


# members at the edges of the batch kernels (4 waves up to ld = 1024, 8 up to 2048; 2050 runs in grouped
# launches), of different sizes, against the grouped dense kernel
@pytest.mark.parametrize("n_wp", [1, 2, 4])
def test_batch_series_matches_terms(ctx, n_wp):
    sizes = [5, 64, 130, 960, 1024, 1025, 1100, 2048, 2050]
    out = []
    for family in (-1, 0):
        hip.force_batch_family(2 * n_wp, family)
        try:
            systems = []
            for N in sizes:
                rng = np.random.default_rng(N)
                a, b = rng.normal(size=(2, N, N)) / np.sqrt(N)
                s = hip.System(ctx, n_orb=N, n_wp=n_wp)
                s.load_operators(np.eye(N) + 0.02 * (a + a.T), 8.0 * (b + b.T) - 10.0 * np.eye(N))
                for w in range(n_wp):
                    c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
                    s.set_initial_state(w, c, c)
                systems.append(s)
            batch = hip.Batch(ctx, systems)
            batch.propagate(0.0, DT)
            batch.propagate_steps(12, DT)
            out.append([[s.wavepacket(w)[1] for w in range(n_wp)] for s in systems])
            batch.close()
            for s in systems:
                s.close()
        finally:
            hip.force_batch_family(2 * n_wp, -1)
    for N, x, y in zip(sizes, *out):
        for w in range(n_wp):
            assert np.linalg.norm(x[w] - y[w]) <= 1e-11 * np.linalg.norm(y[w]), N


# 4 waves per workgroup up to ld = 2048 (1920 for 4 wavepackets): every count of groups per wave from 18 on,
# with and without part of the operator in LDS
@pytest.mark.parametrize("n_wp,sizes", [(1, [1100, 1409, 1537, 1700, 1985, 2048]), (2, [1088, 1473, 1600, 1793, 2000]),
                                        (4, [1150, 1280, 1408, 1530, 1660, 1792, 1920, 1921])])
def test_batch_series_four_waves(ctx, n_wp, sizes):
    out = []
    for family in (-1, 0):
        hip.force_batch_family(2 * n_wp, family)
        try:
            systems = []
            for N in sizes:
                rng = np.random.default_rng(N)
                b = rng.normal(size=(N, N)) / np.sqrt(N)
                s = hip.System(ctx, n_orb=N, n_wp=n_wp)
                s.load_operators(np.eye(N), 8.0 * (b + b.T) - 10.0 * np.eye(N))
                for w in range(n_wp):
                    c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
                    s.set_initial_state(w, c, c)
                systems.append(s)
            batch = hip.Batch(ctx, systems)
            batch.propagate_steps(4, DT)
            out.append([[s.wavepacket(w)[1] for w in range(n_wp)] for s in systems])
            batch.close()
            for s in systems:
                s.close()
        finally:
            hip.force_batch_family(2 * n_wp, -1)
    for N, x, y in zip(sizes, *out):
        for w in range(n_wp):
            assert np.linalg.norm(x[w] - y[w]) <= 1e-11 * np.linalg.norm(y[w]), N


# edges of the sizes whose data are their own flags (2816 at R = 1 and 2, 2304 at 4, 2048 at 8), and counts of
# columns that leave part of a lane's share unwritten
@pytest.mark.parametrize("N,R", [(385, 4), (448, 1), (641, 8), (1024, 2), (1409, 4), (1990, 1), (2047, 8), (2304, 4),
                                 (2305, 4), (2816, 2), (2816, 1), (2817, 2)])
def test_series_without_flags(ctx, operator, N, R):
    print(f"[gpu] series without flags, N={N}, R={R}", flush=True)
    a, ka = _apply(ctx, operator, N, R, -1)
    b, kb = _apply(ctx, operator, N, R, 18 if R <= 8 else 15)
    assert ka == kb
    assert np.linalg.norm(a[:N] - b[:N]) <= 1e-11 * np.linalg.norm(b[:N])


@pytest.mark.parametrize("n_wp,N", [(3, 500), (3, 1500), (3, 2100), (1, 300), (2, 2304)])
def test_steps_without_flags(ctx, operator, n_wp, N):
    """Several long series one after another on one system (stale ring slots of the last one), R = 2, 4 and 6."""
    print(f"[gpu] steps without flags, N={N}, n_wp={n_wp}", flush=True)
    out = []
    for variant in (-1, 9):
        hip.force_matvec_variant(variant)
        try:
            s = hip.System(ctx, n_orb=N, n_wp=n_wp)
            s.load_operators(np.eye(N), operator[:N, :N] * (34.0 / np.sqrt(8.0 * N)))
            rng = np.random.default_rng(N)
            for w in range(n_wp):
                c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
                s.set_initial_state(w, c, c)
            for m in (1, 7, 3, 10):
                s.propagate_steps(m, DT)
            out.append(np.stack([s.wavepacket(w)[1] for w in range(n_wp)]))
            s.close()
        finally:
            hip.force_matvec_variant(-1)
    assert np.linalg.norm(out[0] - out[1]) <= 1e-11 * np.linalg.norm(out[1])
