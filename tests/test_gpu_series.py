"""Multi-step Chebyshev series (dh_propagate_steps): coefficients and accumulators."""
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
