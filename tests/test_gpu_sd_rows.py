"""The steepest descent's fused row passes at the row lengths and view sizes
where their layout changes (a row in one thread, in part of a wavefront, in
one and in two wavefronts; several rows and several views in a workgroup),
against the FP64 oracle and with test_gpu_pcmbir.py's tolerances, and against
the separate passes (option fft_reg 0) for the stopping rule.
"""
import numpy as np
import pytest

from test_gpu_pcmbir import LAM, phase_problems, rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views,rows,cols", [
    (3, 4, 8), (37, 2, 16), (5, 2, 64), (2, 8, 1024), (3, 64, 512), (1, 512, 32), (2, 16, 4)])
def test_fused_rows_match_oracle(views, rows, cols):
    from phasecon_amd.pcmbir import PhaseRetrieval
    pps, win, y, D, Lam, v, w, om = phase_problems(views, rows, cols, 7, True)
    print(f"{views} views of {rows}x{cols}", flush=True)
    ctx = PhaseRetrieval(views, rows, cols, 1.0, 1.0, LAM, 1e5, win)
    ctx.set_problem(y, D, Lam, v, w, None, 0.7)
    iters, upd = ctx.sd_run(5, 0.0)
    gw, gom = ctx.state()
    ctx.close()
    assert list(iters) == [5] * views
    for k, pp in enumerate(pps):
        ow, oom, _, u = pp.sd_run(om[k], w[k], 5, 0.0)
        assert rel_rms(gw[k], ow) < 1e-4
        assert rel_rms(gom[k], oom) < 1e-4
        assert upd[k] == pytest.approx(u, rel=1e-3)


@pytest.mark.parametrize("views,rows,cols", [(9, 16, 16), (4, 8, 1024)])
def test_views_stop_on_their_own(views, rows, cols):
    """Views that stop at different iterations: the counts, and each view's w
    unchanged after its last one (the host reads the flags one iteration
    late)."""
    from phasecon_amd.pcmbir import PhaseRetrieval
    pps, win, y, D, Lam, v, w, om = phase_problems(views, rows, cols, 11, False)
    Lam = Lam * (1.0 + np.arange(views))[:, None, None]  # other conditioning per view
    for k, pp in enumerate(pps):
        pp.Lam = Lam[k]
    ctx = PhaseRetrieval(views, rows, cols, 1.0, 1.0, LAM, 1e5, win)
    ctx.set_problem(y, D, Lam, v, w, om, 0.7)
    iters, _ = ctx.sd_run(40, 1.0)
    gw, gom = ctx.state()
    want = [pp.sd_run(om[k], w[k], 40, 1.0) for k, pp in enumerate(pps)]
    print(f"iterations {list(iters)}, oracle {[q[2] for q in want]}", flush=True)
    assert list(iters) == [q[2] for q in want]
    assert len(set(iters)) > 1
    for k, q in enumerate(want):
        assert rel_rms(gw[k], q[0]) < 1e-4
        assert rel_rms(gom[k], q[1]) < 1e-4
    # the next run starts all views again
    assert (ctx.sd_run(2, 0.0)[0] == 2).all()
    ctx.close()
