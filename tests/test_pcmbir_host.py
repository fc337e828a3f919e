"""The phase retrieval's host side against a stand-in for the HIP runtime
(hip_stub.py): what a failed allocation leaves behind, and what a long descent
holds."""
import os

import numpy as np
import pytest

import hip_stub

pytestmark = pytest.mark.skipif(not os.path.exists(hip_stub.HIPCC), reason="no hipcc")
SHAPE = (2, 16, 32)


@pytest.fixture
def L(monkeypatch):
    return hip_stub.use(monkeypatch)


def _context():
    from phasecon_amd.pcmbir import PhaseRetrieval
    return PhaseRetrieval(*SHAPE, 1.0, 1.0, 1e-4, 1e5)


def _problem(pr):
    a = np.ones(SHAPE, np.complex64)
    pr.set_problem(a, a, np.float32(1), a, a, None, 0.5)


# every call that allocates a group of buffers, and how many there are
@pytest.mark.parametrize("call,n", [
    (_problem, 13),
    (lambda pr: pr.set_tomo_target(0.5, np.ones(SHAPE, complex)), 2),
    (lambda pr: pr.paganin(np.ones(SHAPE, complex), np.ones(SHAPE, complex), 10.0, 1.0), 8)])
def test_a_group_of_buffers_is_whole_or_absent(L, call, n):
    """Whichever buffer fails: the call after it allocates the whole group and
    no launch has run without it."""
    live0 = L.stub_live()
    for after in range(n):
        pr = _context()
        live, runs = L.stub_live(), L.stub_launches()
        L.stub_fail_malloc(after)
        for _ in range(2):                      # the second: still no memory
            with pytest.raises(RuntimeError):
                call(pr)
        assert L.stub_launches() == runs
        L.stub_fail_malloc(-1)
        call(pr)
        assert L.stub_live() == live + n
        pr.close()
        assert L.stub_live() == live0


@pytest.mark.parametrize("fft_reg", [0, 1])
@pytest.mark.parametrize("thresh", [0.0, 1e-9])
def test_a_long_descent_holds_no_more_events(L, fft_reg, thresh):
    """The transforms' event pairs do not grow with the iterations."""
    pr = _context()
    pr.option("fft_reg", fft_reg)
    _problem(pr)
    pr.sd_run(1000, thresh)
    held = L.stub_live_events()
    pr.sd_run(2000, thresh)
    assert L.stub_live_events() == held
    pr.close()
    assert L.stub_live_events() == 0
