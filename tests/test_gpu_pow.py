"""The FP64 prior costs over the range of differences and exponents their
power function sees, against the oracle (libm's pow): sums of positive terms,
each within a few units in the last place, so 1e-13 of the total.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [1.0, 1.2, 1.5, 1.99, 2.0])
def test_prior_cost_over_magnitudes(p):
    """Differences from 1e-20 to 1e6 (and exact zeros, and denormals)."""
    from oracle.oracle import Oracle
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import make_scan
    scan = make_scan("ch4d_small", seed=1, p_s=p, p_t=p)
    st, o = Stage(scan), Oracle(scan)
    rng = np.random.default_rng(int(10 * p))
    for lo, hi in ((-20, -10), (-10, 0), (0, 6), (-44, -38)):
        x = (10.0 ** rng.uniform(lo, hi, st.shape_x) * rng.choice([-1, 0, 1], st.shape_x))
        x = x.astype(np.float32)
        st.set_object(x)
        st.init_error()
        got = st.cost()[2]
        e = np.zeros(o.y.shape)
        want = o.cost(e, x.astype(np.float64))[1][1]
        print(f"p {p}, 1e{lo}..1e{hi}: {got:.17g} vs {want:.17g}", flush=True)
        assert abs(got - want) <= 1e-13 * want
    st.close()
