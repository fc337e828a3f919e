"""The MBIR library's host side against a stand-in for the HIP runtime
(hip_stub.py): what a failed allocation leaves behind, the grids of launches
over many frames, the pinned memory of large copies, and the projector's
exchanged object."""
import os
import threading

import numpy as np
import pytest

import hip_stub

pytestmark = pytest.mark.skipif(not os.path.exists(hip_stub.HIPCC), reason="no hipcc")


@pytest.fixture
def L(monkeypatch):
    return hip_stub.use(monkeypatch)


def _scan(cols=16):
    from phasecon_amd.synth import geometry_scan
    return geometry_scan(4, cols, 6)


def _stage(**kw):
    from phasecon_amd.mbir import Stage
    return Stage(_scan(), **kw)


def _built():
    st = _stage()
    st.build_amatrix()
    return st


def _half():
    st = _built()
    st.option("afp16", 1)
    return st


def _swept():
    st = _built()
    st.icd(1, 1)
    st.option("tile", 4)
    return st


def _tomo():
    from phasecon_amd.mbir import TomoStage, tomo_prior
    p = tomo_prior((2e-7, 1e-3, 0.01, 0.01), (2e-10, 1e-3, 0.01, 0.01), 1, 6.0, 1.0,
                   delta_over_beta=50.0, mu=0.5, alpha=1.5)
    st = TomoStage(_scan(), p)
    z = np.zeros(st.shape_e, np.float32)
    st.init_errors(z, z)
    return st


def _admm(st):
    z = np.zeros(st.shape_e)
    st.admm_init(z, z)


# every call that allocates a group of buffers: the context it is made on, how
# many there are, and a kernel that reads them
@pytest.mark.parametrize("make,call,n,kernel", [
    (_stage, lambda st: st.build_amatrix(), 2, "k_amatrix"),
    (_half, lambda st: st.build_amatrix(), 2, "k_aquant"),
    (_built, lambda st: st.option("nhicd", 1), 2, "k_vsc"),
    (_built, lambda st: st.icd(1, 1), 3, "k_sweep"),
    (_swept, lambda st: st.icd(1, 1), 3, "k_sweep"),
    (_built, lambda st: st.cost(), 1, "k_data_cost"),
    (_tomo, _admm, 5, "k_fwdproj")])
def test_a_group_of_buffers_is_whole_or_absent(L, make, call, n, kernel):
    """Whichever buffer fails: the call after it allocates the whole group and
    no kernel has run without it."""
    live0 = L.stub_live()
    whole = make()
    call(whole)
    live = L.stub_live()
    whole.close()
    for after in range(n):
        st = make()
        L.stub_clear_log()
        L.stub_fail_malloc(after)
        for _ in range(2):                      # the second: still no memory
            with pytest.raises(RuntimeError):
                call(st)
        assert not any(kernel in k[0] for k in hip_stub.launches(L))
        L.stub_fail_malloc(-1)
        call(st)
        assert L.stub_live() == live
        st.close()
        assert L.stub_live() == live0


def test_a_tile_whose_lists_failed_is_not_kept(L):
    """Back at the tile of the last sweep after a failed one: its lists are
    made again, not taken for there."""
    st = _built()
    st.icd(1, 1)
    st.option("tile", 4)
    L.stub_fail_malloc(0)
    with pytest.raises(RuntimeError):
        st.icd(1, 1)
    st.option("tile", 16)
    L.stub_clear_log()
    with pytest.raises(RuntimeError):
        st.icd(1, 1)
    assert not hip_stub.launches(L)
    L.stub_fail_malloc(-1)
    st.icd(1, 1)
    st.close()


def test_grids_of_many_frames(L):
    """Frames beyond what a grid's second and third axis hold (65535): every
    launch of the projections puts them on the first."""
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import geometry_scan
    n = 66000
    s = geometry_scan(1, 16, n)
    s["recon_num"], s["recon_times"] = n, np.arange(n + 1).astype(np.float32)
    st = Stage(s)
    st.build_amatrix()
    st.init_error()
    st.backproject(np.zeros(st.shape_e, np.float32))
    st.close()
    runs = hip_stub.launches(L)
    assert {k for k in ("k_fwdproj", "k_backproj") if any(k in r[0] for r in runs)} \
        == {"k_fwdproj", "k_backproj"}
    for name, x, y, z, threads in runs:
        assert y <= 65535 and z <= 65535 and x * threads < 1 << 32, name


def _large():
    from phasecon_amd.mbir import Stage
    from phasecon_amd.synth import geometry_scan
    return Stage(geometry_scan(33, 256, 2))     # an object of 8.25 MiB


def _round_trip(st, seed):
    x = np.random.default_rng(seed).random(st.shape_x, np.float32)
    st.set_object(x)
    return np.array_equal(st.get_object(), x)


def test_contexts_share_the_pinned_slots(L):
    """Contexts one after another share one set of slots, concurrent copies pin
    at most four, and the last context gives them back; without pinned memory a
    copy goes without."""
    pins, live, events = L.stub_pins(), L.stub_live_pins(), L.stub_live_events()
    sts = [_large() for _ in range(3)]
    L.stub_fail_pin(1)
    assert _round_trip(sts[0], 0)
    L.stub_fail_pin(0)
    assert L.stub_pins() == pins
    assert all(_round_trip(st, i) for i, st in enumerate(sts))
    assert L.stub_pins() == pins + 1 and L.stub_live_pins() == live + 1
    sts.pop().close()
    assert _round_trip(sts[0], 5) and L.stub_pins() == pins + 1
    for st in sts:
        st.close()
    assert L.stub_live_pins() == live and L.stub_live_events() == events
    sts, ok = [_large() for _ in range(6)], []
    th = [threading.Thread(target=lambda st=st: ok.append([_round_trip(st, i) for i in range(8)]))
          for st in sts]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert ok == [[True] * 8] * 6
    assert 1 <= L.stub_live_pins() - live <= 4
    for st in sts:
        st.close()
    assert L.stub_live_pins() == live and L.stub_live_events() == events


def test_the_exchanged_object_takes_no_room_of_its_own(L):
    """The error sinogram and the cost exchange x and y in the staging buffer;
    A x alone allocates for it, and nothing is exchanged where no view's lines
    run along y, nor for an object of at most 64^2 columns."""
    from phasecon_amd.mbir import Stage
    st = Stage(_scan(65))
    st.build_amatrix()
    live = L.stub_live()
    st.init_error()
    assert L.stub_live() == live
    assert any("k_swap_xy" in r[0] for r in hip_stub.launches(L))
    st.forward_project(np.zeros(st.shape_x, np.float32))
    assert L.stub_live() == live + 1
    st.close()
    L.stub_clear_log()
    flat = _scan(65)
    flat["angles"] = np.linspace(-0.7, 0.7, 6).astype(np.float32)
    for s in (flat, _scan(64)):
        st = Stage(s)
        st.init_error()
        st.forward_project(np.zeros(st.shape_x, np.float32))
        st.close()
    runs = [r[0] for r in hip_stub.launches(L)]
    assert any("k_fwdproj" in r for r in runs) and not any("k_swap_xy" in r for r in runs)
