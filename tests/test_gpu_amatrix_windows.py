"""The A build at the edges of its block: entries that do not fill the last
block, and windows up to the widest (W = 33), against the oracle: first bins
exact, values within the rounding to 32 bits of the detector response and of
the value, 2^-23 of the largest.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,views,mult", [(6, 7, 1), (21, 13, 1), (48, 11, 4), (64, 9, 16)])
def test_windows_match_oracle(cols, views, mult):
    from oracle.oracle import Oracle
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import geometry_scan
    scan = geometry_scan(1, cols, views)
    st, o = Stage(scan, mult_xy=mult), Oracle(scan, mult_xy=mult)
    st.build_amatrix()
    first, val = st.get_amatrix()
    ofirst, oval = o.amatrix_all()
    print(f"{cols} columns, {views} views, mult {mult}: {val.shape}", flush=True)
    assert np.array_equal(first, ofirst)
    assert np.abs(val - oval).max() <= 2.0 ** -23 * np.abs(oval).max()
    st.close()
