"""Launches whose waits run out: the result is marked, and the step, batch member or bounds are formed again by one
launch per term (or step), with the same spectral bounds.  The hook makes every wave give up at once.

The repeat evaluates the same series with other kernels: 1e-11 of the norm as in the comparison of the two."""
import numpy as np
import pytest

from dynemol_amd import hip

pytestmark = pytest.mark.gpu
DT = 5.0e-4


@pytest.fixture(params=[False, True], ids=["", "give up"])
def both(request):
    """Each test runs its case without and with waits that run out; the first run's result is the reference."""
    hip.force_give_up(request.param)
    yield request.param
    hip.force_give_up(False)


@pytest.fixture(scope="module")
def seen():
    return {}


def _system(ctx, N, n_wp, zero=()):
    rng = np.random.default_rng(N)
    b = rng.normal(size=(N, N)) / np.sqrt(N)
    s = hip.System(ctx, n_orb=N, n_wp=n_wp)
    s.load_operators(np.eye(N), 8.0 * (b + b.T) - 10.0 * np.eye(N))
    for w in range(n_wp):
        c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
        s.set_initial_state(w, c * (w not in zero), c * (w not in zero))
    return s


def _close(seen, key, value):
    ref = seen.setdefault(key, value)
    assert np.linalg.norm(value - ref) <= 1e-11 * np.linalg.norm(ref)


# data as flags and flags, one and two column sets, one real column per lane
@pytest.mark.parametrize("N,n_wp", [(500, 1), (900, 2), (700, 4), (2900, 2)])
def test_steps(both, seen, N, n_wp):
    print(f"[gpu] give up: steps, N={N}, n_wp={n_wp}, {both}", flush=True)
    with hip.Context(0) as ctx:
        s = _system(ctx, N, n_wp)
        terms = s.propagate(0.0, DT)
        assert s.stats()["retries"] == (1 if both else 0)
        assert seen.setdefault(("terms", N, n_wp), terms) == terms  # the bounds were not widened
        pops, erg, _ = s.propagate_steps(4, DT)
        assert s.stats()["retries"] == (2 if both else 0)
        _close(seen, ("state", N, n_wp), np.stack([s.wavepacket(w) for w in range(n_wp)]))
        _close(seen, ("pops", N, n_wp), pops)
        _close(seen, ("erg", N, n_wp), erg)
        s.close()


@pytest.mark.parametrize("n_wp", [1, 2, 4])
def test_batch(both, seen, n_wp):
    """Members with a zero wavepacket, and one with nothing else."""
    print(f"[gpu] give up: batch, n_wp={n_wp}, {both}", flush=True)
    with hip.Context(0) as ctx:
        systems = [_system(ctx, 520, n_wp), _system(ctx, 1300, n_wp, zero=range(1, n_wp)),
                   _system(ctx, 640, n_wp, zero=range(n_wp))]
        batch = hip.Batch(ctx, systems)
        batch.propagate(0.0, DT)
        batch.propagate_steps(4, DT)
        for i, s in enumerate(systems):
            _close(seen, ("batch", n_wp, i), np.stack([s.wavepacket(w) for w in range(n_wp)]))
            assert (s.stats()["retries"] > 0) == both
        batch.close()
        for s in systems:
            s.close()


def test_bounds(both):
    """The bounds of a launch that gave up are those formed step by step."""
    print(f"[gpu] give up: bounds, {both}", flush=True)
    with hip.Context(0) as ctx:
        s = _system(ctx, 700, 1)
        got = s.bounds()
        s.close()
        hip.force_give_up(False)
        s = hip.System(ctx, n_orb=700, n_wp=1)
        s.set_one_launch_bounds(False)
        rng = np.random.default_rng(700)
        b = rng.normal(size=(700, 700)) / np.sqrt(700)
        s.load_operators(np.eye(700), 8.0 * (b + b.T) - 10.0 * np.eye(700))
        step_by_step = s.bounds()
        s.close()
    assert np.isfinite(got).all()
    if both:
        assert np.array_equal(got, step_by_step)


def _apply(ctx, N, R, bounds, dt, variant=-1):
    ld = (N + 63) // 64 * 64
    rng = np.random.default_rng(N)
    x = rng.normal(size=(N, N))
    H = np.zeros((ld, ld))
    H[:N, :N] = (x + x.T) * (17.0 / np.sqrt(2.0 * N))  # half width 34
    phi = np.zeros((ld, R), dtype=complex)
    phi[:N] = (rng.normal(size=(N, R)) + 1j * rng.normal(size=(N, R))) / np.sqrt(2.0 * N)
    bufs = [hip.DeviceBuffer(H.nbytes), hip.DeviceBuffer(phi.nbytes), hip.DeviceBuffer(hip.chebyshev_work_bytes(N, R))]
    try:
        bufs[0].upload(H)
        bufs[1].upload(phi)
        hip.force_matvec_variant(variant)
        k = hip.chebyshev_apply(ctx, N, bufs[0].ptr, ld, bounds, dt, R, bufs[1].ptr, bufs[2].ptr, bufs[2].nbytes)
        out = bufs[1].download((ld, R), np.complex128)[:N]
    finally:
        hip.force_matvec_variant(-1)
        for b in bufs:
            b.close()
    E, V = np.linalg.eigh(H[:N, :N])
    exact = V @ (np.exp(-1j * E * dt / hip.H_BAR)[:, None] * (V.T @ phi[:N]))
    return out, k, exact


def test_apply(both, seen):
    print(f"[gpu] give up: caller's operator, {both}", flush=True)
    with hip.Context(0) as ctx:
        out, k, exact = _apply(ctx, 800, 4, [-36.0, 36.0], DT)
    assert seen.setdefault("apply terms", k) == k
    assert np.linalg.norm(out - exact) <= 1e-9 * np.linalg.norm(exact)


@pytest.mark.parametrize("N,R,variant", [(800, 4, -1), (800, 4, 1), (100, 4, -1)])
def test_too_narrow_bounds_that_overflow(N, R, variant):
    """A long step on bounds of 0.6 of the half width: the first series overflow.  They tell of the bounds, unless
    the series ran in one launch, and three widenings by 1.25 are enough, in one launch (800), with a forced
    kernel and at a size that runs term by term."""
    print(f"[gpu] narrow bounds, N={N}, variant {variant}", flush=True)
    with hip.Context(0) as ctx:
        out, _, exact = _apply(ctx, N, R, [-20.4, 20.4], 0.03, variant)
    assert np.linalg.norm(out - exact) <= 1e-9 * np.linalg.norm(exact)
