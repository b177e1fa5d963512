"""dh_system_bytes_prec, by which the server admits requests, covers what a system holds on the device."""
import numpy as np
import pytest
import torch

from dynemol_amd import hip

pytestmark = pytest.mark.gpu
DT = 5.0e-4
SLACK = 4 << 20  # allocations are rounded up to 2 MiB pages: about 30 small ones share a few


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info(0)[0]


def _system(ctx, N, n_wp):
    rng = np.random.default_rng(N)
    b = rng.normal(size=(N, N)) * (8.0 / np.sqrt(N))
    s = hip.System(ctx, n_orb=N, n_wp=n_wp)
    s.load_operators(np.eye(N), b + b.T)
    c = (rng.normal(size=N) + 1j * rng.normal(size=N)) / np.sqrt(2.0 * N)
    for w in range(n_wp):
        s.set_initial_state(w, c, c)
    return s


@pytest.mark.parametrize("N,n_wp", [(416, 2), (1700, 4), (2304, 8), (1000, 16)])
def test_footprint_after_steps(N, n_wp):
    print(f"[gpu] footprint, N={N}, n_wp={n_wp}", flush=True)
    with hip.Context(0) as ctx:
        s = _system(ctx, N, n_wp)  # the context's workspace and the kernels' own memory
        s.propagate_steps(8, DT)
        s.close()
        before = _free()
        systems = [_system(ctx, N, n_wp) for _ in range(4)]
        for s in systems:
            s.propagate_steps(8, DT)
        held = (before - _free()) / 4
        for s in systems:
            s.close()
    print(f"  held {held / 2**20:.1f} MiB, counted {hip.system_bytes(N, n_wp) / 2**20:.1f} MiB", flush=True)
    assert held <= hip.system_bytes(N, n_wp) + SLACK


def test_long_calls_give_their_block_back():
    """80000 steps take 5 MB, more than stays with a system, and their results do not fit the pinned buffer."""
    print("[gpu] footprint after a long call", flush=True)
    with hip.Context(0) as ctx:
        s = _system(ctx, 64, 1)
        out = s.propagate_steps(80000, 1e-9)
        a = s.wavepacket(0)
        s.close()
        s = _system(ctx, 64, 1)
        parts = [s.propagate_steps(20000, 1e-9) for _ in range(4)]
        b = s.wavepacket(0)
        s.close()
    assert np.array_equal(out[0], np.concatenate([p[0] for p in parts]))
    assert np.array_equal(out[1], np.concatenate([p[1] for p in parts]))
    assert np.array_equal(a, b)
