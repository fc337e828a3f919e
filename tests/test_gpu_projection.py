"""The forward projection (gathered per detector bin), the back-projection and
the ramp filter at sizes where their chunks are not full, against numpy on
the system matrix the library built (itself bit-checked against the oracle in
test_gpu_mbir.py).

Tolerances: A is stored in FP32 (2^-24 per value), the projection's sums are
FP64 and rounded once, so 1e-6 of the largest value; the back-projection sums
up to 40 x 9 FP32 terms, 1e-5.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scan(rows, cols, views, frames, rot=None):
    from phasecon_amd.synth import geometry_scan
    s = geometry_scan(rows, cols, views * frames)
    s["recon_num"] = frames
    s["recon_times"] = (np.arange(frames + 1) * views).astype(np.float32)
    s["angles"] = (np.random.default_rng(cols).permutation(views * frames) * np.pi /
                   (views * frames) - 0.3).astype(np.float32)
    if rot is not None:
        s["rot_center"] = rot
    return s


def _dense(st, x, v):
    """A x [N_p][N_r][N_t] and A^T v [N_time][N_z][N_y][N_x] in FP64."""
    first, val = st.get_amatrix()
    g = st.g
    zo, nz = g.mult_z, g.N_z
    ax = np.zeros((g.N_p, g.N_r + st.W, g.N_t))
    bt = np.zeros((g.N_time, g.N_y * g.N_x, nz))
    vp = np.concatenate([v, np.zeros((g.N_p, st.W, g.N_t), v.dtype)], 1).astype(np.float64)
    for f in range(g.N_time):
        xf = x[f].reshape(nz, -1).T.astype(np.float64)
        for s in range(st.frame_ptr[f], st.frame_ptr[f + 1]):
            p, hit = st.frame_views[s], first[:, s] >= 0
            for k in range(st.W):
                r, a = first[hit, s] + k, val[hit, s, k].astype(np.float64)
                np.add.at(ax[p], r, np.repeat(a[:, None] * xf[hit], zo, 1))
                bt[f][hit] += a[:, None] * vp[p][r].reshape(-1, nz, zo).sum(2)
    return ax[:, :g.N_r], bt.transpose(0, 2, 1).reshape(g.N_time, nz, g.N_y, g.N_x)


def _check(st, seed):
    rng = np.random.default_rng(seed)
    x = rng.random(st.shape_x).astype(np.float32)
    x[rng.random(st.shape_x) < 0.2] = 0.0
    v = rng.standard_normal(st.shape_e).astype(np.float32)
    st.build_amatrix()
    want, bt = _dense(st, x, v)
    ax = st.forward_project(x)
    assert np.abs(ax - want).max() <= 1e-6 * np.abs(want).max()
    st.set_object(x)
    st.init_error()
    e = st.get_error()
    assert np.abs(e - (st.y - want)).max() <= 1e-6 * np.abs(want).max()
    c = st.cost(fresh=True)[1]   # huber_T 1e5: the quadratic branch
    data = 0.5 * np.sum((st.y - want) ** 2 * st.w)
    assert abs(c - data) <= 1e-6 * data
    back = st.backproject(v)
    assert np.abs(back - bt).max() <= 1e-5 * np.abs(bt).max()


# detectors below, at and above a workgroup's bins (32 to 512); one to 40
# slices; rows per slice 1, 2 and 3; an off-centre axis, where columns miss the
# detector.  Few workgroups take 4 slices each, whatever there are; from 256 on
# 8 or 16: the second line has both, below, at and above a chunk
@pytest.mark.parametrize("rows,cols,views,frames,mxy,mz,rot", [
    (1, 16, 7, 1, 1, 1, None), (3, 32, 5, 2, 1, 1, None), (8, 66, 9, 3, 1, 1, 20.0),
    (10, 64, 4, 1, 2, 2, None), (9, 60, 6, 2, 3, 3, None), (24, 48, 5, 2, 4, 1, 30.5),
    (40, 34, 3, 1, 1, 1, None), (4, 520, 3, 1, 1, 1, None), (17, 130, 2, 2, 1, 1, None),
    (7, 20, 130, 2, 1, 1, None), (8, 20, 130, 2, 1, 1, 7.5), (10, 20, 70, 2, 1, 1, None),
    (13, 24, 130, 2, 1, 1, None), (16, 24, 130, 2, 2, 1, None), (20, 20, 65, 2, 1, 1, 11.0),
    (34, 24, 130, 2, 1, 2, None), (3, 70, 4, 2, 1, 1, None), (10, 70, 65, 2, 1, 1, 31.0),
    (17, 66, 65, 2, 1, 1, None)])
def test_projections_match_the_system_matrix(rows, cols, views, frames, mxy, mz, rot):
    from phasecon_amd.mbir import Stage
    print(f"rows {rows}, cols {cols}, views {views} x {frames}, mult {mxy}/{mz}", flush=True)
    st = Stage(_scan(rows, cols, views, frames, rot), mult_xy=mxy, mult_z=mz)
    _check(st, rows + cols)
    st.close()


# every view's image lines along x, along y; objects that are exchanged for the
# latter (above 64^2 columns) and that are not
@pytest.mark.parametrize("cols", [48, 64, 65, 100])
@pytest.mark.parametrize("lo,hi", [(-0.78, 0.78), (0.79, 2.35)])
def test_views_of_one_axis(lo, hi, cols):
    from phasecon_amd.mbir import Stage
    s = _scan(6, cols, 5, 2)
    s["angles"] = np.linspace(lo, hi, 10).astype(np.float32)
    print(f"angles {lo} to {hi}, cols {cols}", flush=True)
    st = Stage(s)
    _check(st, 9)
    st.close()


def test_entries_that_a_does_not_hold():
    """A keeps positive responses only: where the response table is zero or
    negative the projection adds nothing, not even of an infinite voxel."""
    from phasecon_amd import lib
    from phasecon_amd.mbir import Stage, _p
    st = Stage(_scan(5, 40, 6, 2))
    st.L.mbir_hip_destroy(st.h)
    st.H[:, 20:30] = 0.0
    st.H[:, 40:] = -np.abs(st.H[:, 40:]) - 0.1
    h = C.c_void_p()
    lib.check(st.L.mbir_hip_create(C.byref(h), C.byref(st.g), _p(st.H), _p(st.cos), _p(st.sin),
                                   _p(st.frame_ptr), _p(st.frame_views), _p(st.y), _p(st.w), None,
                                   _p(st.mask)), "mbir_hip_create")
    st.h = h
    print("response table with zeros and negative values", flush=True)
    _check(st, 4)
    x = np.random.default_rng(4).random(st.shape_x).astype(np.float32)
    want, _ = _dense(st, x, st.y)
    x[0, 2, 17, 22] = np.inf
    first, val = st.get_amatrix()
    ax = st.forward_project(x)
    st.close()
    c = 17 * st.g.N_x + 22
    hit = np.zeros(st.shape_e, bool)
    for s in range(st.frame_ptr[0], st.frame_ptr[1]):
        for k in np.nonzero(val[c, s])[0]:
            hit[st.frame_views[s], first[c, s] + k, 2] = True
    assert np.isinf(ax[hit]).all() and hit.any()
    assert np.abs(ax - want)[~hit].max() <= 1e-6 * np.abs(want).max()


# 4, 8 and 16 slices per workgroup
@pytest.mark.parametrize("rows,cols,views", [(5, 40, 6), (7, 24, 130), (20, 24, 65)])
@pytest.mark.parametrize("factor", [1.7, 0.6])
def test_other_response_tables(factor, rows, cols, views):
    """A response table over another width than the usual one (the window of
    the A rule then cuts it, or a bin meets more voxels of a line)."""
    from phasecon_amd import lib
    from phasecon_amd.mbir import Stage, _p
    st = Stage(_scan(rows, cols, views, 2))
    st.L.mbir_hip_destroy(st.h)
    st.g.OffsetR *= factor
    h = C.c_void_p()
    lib.check(st.L.mbir_hip_create(C.byref(h), C.byref(st.g), _p(st.H), _p(st.cos), _p(st.sin),
                                   _p(st.frame_ptr), _p(st.frame_views), _p(st.y), _p(st.w), None,
                                   _p(st.mask)), "mbir_hip_create")
    st.h = h
    print(f"OffsetR x {factor}, rows {rows}, cols {cols}, views {views} x 2", flush=True)
    _check(st, 3)
    st.close()


# the last: more channels than the ramp filter stages
@pytest.mark.parametrize("rows,cols,views,mxy", [
    (1, 32, 3, 1), (20, 50, 4, 1), (17, 400, 2, 1), (2, 6208, 2, 16)])
def test_fbp_matches_numpy(rows, cols, views, mxy):
    """A^T ramp(y) / K with the ramp as a dense FP64 matrix."""
    from phasecon_amd.mbir import Stage
    s = _scan(rows, cols, views, 1)
    s["projections"] = np.random.default_rng(1).random((views, rows, cols)).astype(np.float32)
    st = Stage(s, mult_xy=mxy)
    st.build_amatrix()
    print(f"fbp {rows}x{cols}, {views} views", flush=True)
    out = st.fbp()
    n = np.arange(cols)[:, None] - np.arange(cols)[None, :]
    h = np.where(n == 0, 0.25, np.where(n % 2 != 0, -1.0 / (np.pi * np.where(n == 0, 1, n)) ** 2, 0))
    ramp = lambda v: np.einsum("rq,pqt->prt", h, v.astype(np.float64))  # noqa: E731
    ones = np.broadcast_to(st.mask[None, None].astype(np.float32), st.shape_x)
    am, _ = _dense(st, ones, st.y)
    _, k = _dense(st, ones, ramp(am))
    _, want = _dense(st, ones, ramp(st.y))
    K = k[:, :, st.mask != 0].mean()
    st.close()
    assert np.abs(out - want / K).max() <= 1e-5 * np.abs(want / K).max()
