"""The sweep with its sinogram side on several wavefronts (windows that are
not one load batch of one wavefront), voxel by voxel against the oracle's
restatement of its schedule, as test_gpu_sweep_order.py does for the
benchmark's shapes and with the same tolerance: one launch per tile colour
and frame parity, so the sweep is the oracle's sequential ICD.

Launches of more workgroups than the chip has CUs give the sinogram side two
wavefronts, the largest one: with many frames of one tile per colour they are
just as deterministic; with several tiles of a frame at once (the last test) the
maintained error sinogram stays y - A x and the cost falls.

Non-homogeneous passes rank a tile's columns with all of a workgroup's
threads, 192 or 320 here: test_gpu_nhicd.py's test on such geometries, with
tiles of fewer and of more columns than threads.

Shapes: row counts that are and are not powers of two and above one
wavefront, view counts at both sides of a load batch and not a multiple of
the slots that the wavefronts share.
"""
import numpy as np
import pytest

from test_gpu_sweep_order import TOL, _start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,views", [
    (8, 32, 17), (8, 32, 33),     # just above one wavefront's load batch
    (24, 32, 7), (24, 32, 29),    # 24 rows: 2 groups of 24 lanes
    (12, 32, 20), (34, 16, 17),   # 4 groups of 12, one group of 34
    (80, 16, 11)])                # rows above one wavefront
def test_wide_sweep_matches_oracle_schedule(rows, cols, views, frames=1):
    from oracle.oracle import Oracle
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import make_scan
    scan = make_scan("tall3d", seed=1, rows=rows, cols=cols, views=views * frames, frames=frames)
    o = Oracle(scan)
    T = cols // 2
    print(f"rows {rows}, cols {cols}, views {views} x {frames}", flush=True)
    x0 = _start(o, 20, False)
    st = Stage(scan, tile=T, alpha=1.5)
    st.option("pair_parities", 0)  # the launch order the oracle's model follows
    st.set_object(x0.astype(np.float32))
    st.build_amatrix()
    st.init_error()
    st.icd(1, 21, 4242)
    xg = st.get_object().astype(np.float64)
    eg = st.get_error().astype(np.float64)
    st.close()
    xo = x0.copy()
    eo = o.init_error(xo)
    o.icd_equit_async(xo, eo, 21, T, 1.5, 4242, 0, 0, 0, 8, 0)
    dx = np.abs(xg - xo).max() / np.abs(xo).max()
    de = np.abs(eg - eo).max() / np.abs(o.y).max()
    moved = np.abs(xo - x0).max() / np.abs(xo).max()
    print(f"dx {dx:.3g} de {de:.3g} moved {moved:.3g}", flush=True)
    assert moved > 100 * TOL
    assert dx < TOL
    assert de < TOL


# 260 workgroups in each launch (one per frame of a parity); 1280, as many of
# three wavefronts as the chip holds, and 1320, where the sinogram side goes back
# to one wavefront
@pytest.mark.parametrize("rows,views,frames", [
    (3, 3, 520), (5, 18, 520), (24, 7, 520), (3, 3, 2560), (3, 3, 2640), (5, 18, 2640)])
def test_wide_sweep_of_many_frames_matches_oracle_schedule(rows, views, frames):
    test_wide_sweep_matches_oracle_schedule(rows, 8 if frames > 520 else 12, views, frames)


# four wavefronts (tile 8, 16: 64 and 256 columns, 320 threads), then two
# (70 frames of 4 tiles per colour: 280 workgroups of 192 threads)
@pytest.mark.parametrize("T,frames", [(8, 4), (16, 4), (16, 140)])
def test_nh_pass_of_a_wide_sweep(T, frames):
    from phasecon_amd.synth import make_scan
    from test_gpu_nhicd import test_nh_pass_visits_the_top_columns_of_each_tile as check
    print(f"tile {T}, {frames} frames", flush=True)
    check(make_scan("tall3d", seed=2, rows=3, cols=64, views=7 * frames, frames=frames), 0.3, T)


@pytest.mark.parametrize("rows,views", [(8, 20 * 16), (12, 7 * 16)])
def test_wide_sweep_in_large_launches(rows, views):
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import make_scan
    scan = make_scan("ch4d_small", seed=2, rows=rows, views=views, frames=16)
    print(f"rows {rows}, views {views}", flush=True)
    st = Stage(scan, tile=4, alpha=1.0)   # about 50 tiles per colour x 8 frames
    st.build_amatrix()
    st.init_error()
    costs = [st.cost()[0]]
    for it in range(1, 7):
        st.icd(1, it)
        costs.append(st.cost()[0])
    kept = st.get_error().astype(np.float64)
    st.init_error()
    fresh = st.get_error().astype(np.float64)
    st.close()
    d = np.abs(kept - fresh).max() / np.abs(st.y).max()
    print(f"kept e off by {d:.3g}, costs {costs[0]:.6g} -> {costs[-1]:.6g}", flush=True)
    # six equits of about 200 atomic additions per entry, each rounded to 2^-24
    assert d < 2e-5
    assert costs[-1] < 0.5 * costs[0]


# 16 tiles per colour x 85 frames of a parity: one wavefront on the sinogram
# side, load batches of W = 5 and W = 9
@pytest.mark.parametrize("rows,views,mxy", [(6, 9, 2), (3, 21, 2), (6, 7, 4)])
def test_busy_sweep_of_wide_bins(rows, views, mxy):
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import make_scan
    scan = make_scan("tall3d", seed=4, rows=rows, cols=32 * mxy, views=views * 170, frames=170)
    print(f"rows {rows}, views {views} x 170, mult_xy {mxy}", flush=True)
    st = Stage(scan, mult_xy=mxy, tile=4, alpha=1.0)
    st.build_amatrix()
    st.init_error()
    costs = [st.cost()[0]]
    for it in range(1, 7):
        st.icd(1, it)
        costs.append(st.cost()[0])
    kept = st.get_error().astype(np.float64)
    x, st2 = st.get_object(), Stage(scan, mult_xy=mxy, tile=16, alpha=1.0)
    st.init_error()
    fresh = st.get_error().astype(np.float64)
    st.close()
    # the same equits with few, larger tiles, two wavefronts: near the same object
    st2.build_amatrix()
    st2.init_error()
    for it in range(1, 7):
        st2.icd(1, it)
    c2 = st2.cost()[0]
    st2.close()
    d = np.abs(kept - fresh).max() / np.abs(st.y).max()
    print(f"kept e off by {d:.3g}, costs {costs[0]:.6g} -> {costs[-1]:.6g}, tile 16 {c2:.6g}",
          flush=True)
    # as above; after six equits neither schedule is at the optimum, but both
    # costs are a few per cent of the first, and so is what they differ by
    assert d < 2e-5
    assert np.isfinite(x).all() and costs[-1] < 0.1 * costs[0]
    assert abs(costs[-1] - c2) < 0.02 * costs[0]
