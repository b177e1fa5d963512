"""A batch member's result is the same bits alone and beside larger members.

Members share a launch whose kernel is built for the largest one's groups of 16 columns per wave; the sizes here
are those at which part of the operator is in LDS (from 25, 24 and 23 groups on for 1, 2 and 4 wavepackets), where
the order of a member's sums must not follow the largest one's."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu
DT = 5.0e-4


def _system(ctx, N, n_wp):
    rng = np.random.default_rng(N)
    b = rng.normal(size=(N, N)) / np.sqrt(N)
    s = hip.System(ctx, n_orb=N, n_wp=n_wp)
    s.load_operators(np.eye(N), 8.0 * (b + b.T) - 10.0 * np.eye(N))
    for w in range(n_wp):
        c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
        s.set_initial_state(w, c, c)
    return s


@pytest.mark.parametrize("n_wp,probe,others", [(1, 1590, [1780]), (1, 1700, [2048, 300]), (2, 1500, [1660]),
                                               (2, 1530, [2000, 1800]), (4, 1450, [1590]), (4, 1500, [1920, 700])])
def test_alone_and_beside_larger_members(n_wp, probe, others):
    print(f"[gpu] batch bits N={probe}, n_wp={n_wp} beside {others}", flush=True)
    out = []
    with hip.Context(0) as ctx:
        for sizes in ([probe], [probe] + others):
            systems = [_system(ctx, N, n_wp) for N in sizes]
            batch = hip.Batch(ctx, systems)
            batch.propagate(0.0, DT)
            batch.propagate_steps(3, DT)
            out.append([systems[0].wavepacket(w) for w in range(n_wp)])
            batch.close()
            for s in systems:
                s.close()
    for (bra, ket), (bra2, ket2) in zip(*out):
        assert np.array_equal(ket, ket2)
        assert np.array_equal(bra, bra2)


# one size per instance of the kernels: 2 groups more per wave each time, the last column of the last group missing
@pytest.mark.parametrize("n_wp,largest", [(1, 2048), (2, 2048), (4, 1920)])
def test_no_member_is_redone(n_wp, largest):
    """A member whose norms do not hold is propagated again by other kernels, which would hide a wrong instance."""
    print(f"[gpu] batches of one member, n_wp={n_wp}", flush=True)
    with hip.Context(0) as ctx:
        for N in range(127, largest, 128):
            s = _system(ctx, N, n_wp)
            batch = hip.Batch(ctx, [s])
            batch.propagate(0.0, DT)
            batch.propagate_steps(3, DT)
            retries = s.stats()["retries"]
            batch.close()
            s.close()
            assert retries == 0, N


@pytest.mark.parametrize("n_wp,sizes", [(1, [*range(127, 1024, 128), *range(1279, 4096, 256)]),
                                        (2, [*range(127, 1024, 128), *range(1279, 4096, 256)]),
                                        (4, [*range(127, 1024, 128), *range(1279, 3840, 256)])])
def test_no_step_is_redone(n_wp, sizes):
    """The same for a system on its own (series of one step and of several)."""
    print(f"[gpu] systems on their own, n_wp={n_wp}", flush=True)
    rng = np.random.default_rng(n_wp)
    b = rng.normal(size=(sizes[-1], sizes[-1]))
    b = b + b.T
    with hip.Context(0) as ctx:
        for N in sizes:
            s = hip.System(ctx, n_orb=N, n_wp=n_wp)
            s.load_operators(np.eye(N), b[:N, :N] * (8.0 / np.sqrt(N)))
            for w in range(n_wp):
                c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
                s.set_initial_state(w, c, c)
            s.propagate(0.0, DT)
            s.propagate_steps(3, DT)
            retries = s.stats()["retries"]
            s.close()
            assert retries == 0, N
