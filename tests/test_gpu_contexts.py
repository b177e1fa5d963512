"""Contexts side by side: what a system computes does not depend on the other contexts of the process."""
import threading

import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu
DT = 5.0e-4


def _system(ctx, N, n_wp, one_launch_bounds=True):
    rng = np.random.default_rng(N)
    b = rng.normal(size=(N, N)) / np.sqrt(N)
    s = hip.System(ctx, n_orb=N, n_wp=n_wp)
    s.set_graph(False)
    s.set_one_launch_bounds(one_launch_bounds)
    s.load_operators(np.eye(N), 8.0 * (b + b.T) - 10.0 * np.eye(N))
    for w in range(n_wp):
        c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
        s.set_initial_state(w, c, c)
    return s


@pytest.mark.parametrize("N", [130, 900])
def test_bounds_do_not_depend_on_other_contexts(N):
    print(f"[gpu] bounds with one and with three contexts, N={N}", flush=True)
    bounds = []
    with hip.Context(0) as ctx:
        _system(ctx, N, 1).close()  # kernels chosen
        for others in (0, 2):
            more = [hip.Context(0) for _ in range(others)]
            s = _system(ctx, N, 1)
            bounds.append(s.bounds())
            s.close()
            for c in more:
                c.close()
        s = _system(ctx, N, 1, one_launch_bounds=False)
        step_by_step = s.bounds()
        s.close()
    assert np.array_equal(bounds[0], bounds[1])
    # extreme Ritz values of two summation orders: a few (N + steps) eps of the norm (below 40) per step
    assert np.abs(step_by_step[2:4] - bounds[0][2:4]).max() <= 4.0 * 48 * (N + 48) * np.finfo(float).eps * 40.0


def test_series_of_two_threads_take_turns():
    """Two threads, a context each, whose series want the whole chip: the same bits as one after the other."""
    print("[gpu] series of two threads, N=2100 and 4000", flush=True)
    sizes, steps = [(2100, 2), (4000, 1)], 12
    contexts = [hip.Context(0) for _ in sizes]
    out = []
    for together in (False, True):
        systems = [_system(c, N, w, one_launch_bounds=False) for c, (N, w) in zip(contexts, sizes)]
        failed = []

        def run(s):
            try:
                for _ in range(steps):
                    s.propagate_steps(2, DT)
            except hip.DHError as e:
                failed.append(e)

        if together:
            threads = [threading.Thread(target=run, args=(s,)) for s in systems]
            for t in threads:
                t.start()
            for t in threads:
                t.join()
        else:
            for s in systems:
                run(s)
        assert not failed
        assert [s.stats()["retries"] for s in systems] == [0, 0]
        out.append([np.stack([s.wavepacket(w) for w in range(s.n_wp)]) for s in systems])
        for s in systems:
            s.close()
    for c in contexts:
        c.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
