"""Time steps with a fresh stage 1 (parity=False) against the oracle, the tensors of
level 2 that a caller keeps across them, and the stage evaluated at another state than
the one it overwrites (sodhip_rk_stage_from_f64).  Per-step bar of the other time-loop
tests (FP64 sums reassociate: 1e-12).  A stage from level 1 gives the bits of the stage
in place on a copy of it, in both operator precisions."""
import ctypes as C

import numpy as np
import pytest

from helpers import make_case, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,n,clusters", [(2, 3, 0), (3, 3, 0), (3, 4, 1), (4, 2, 0)])
@pytest.mark.parametrize("dt_mode", ["fixed", "adaptive"])
def test_fresh_stage1(monkeypatch, p, n, clusters, dt_mode):
    from oracle import oracle as O
    from sod2d_amd.device import Context
    from sod2d_amd.solver import TGVParams, TGVRun
    g = make_case(p, n, periodic=True, lengths=(2 * np.pi,) * 3)
    tp, to = TGVParams(), O.tgv_params()
    ic = O.tgv_ic(g.mesh.coord, to)
    if clusters:
        monkeypatch.setenv("SODHIP_STAGE_CLUSTERS", "1")
    ctx = Context(0)
    monkeypatch.delenv("SODHIP_STAGE_CLUSTERS", raising=False)
    run = TGVRun(p, geometry=g, params=tp, initial=ic, ctx=ctx, dt_mode=dt_mode, parity=False)
    orc = O.TGVOracle(p, g, ic, to, parity=False, dt_mode=dt_mode, cfl=(tp.cfl_conv, tp.cfl_diff))
    w = orc.lpoin_w - 1
    for step in range(3):
        run.step()
        orc.step()
        s = run.state()
        for k in ("rho", "q", "E"):
            assert relerr(s[k][w], getattr(orc, k)[1][w]) < 1e-12, (k, step)


@pytest.mark.parametrize("precision,lps", [(8, False), (4, False), (8, True)])
def test_level2_tensors_stay_level2(precision, lps):
    """A caller may take run.rho[1], run.q[1] and run.E[1] once; what it writes there
    at nodes that no working node stands for stays."""
    import torch
    from sod2d_amd.solver import TGVRun
    g = make_case(3, 3, periodic=True, lengths=(2 * np.pi,) * 3)
    run = TGVRun(3, geometry=g, parity=False, dt_mode="fixed", op_precision=precision, lps=lps)
    held = [run.rho[1], run.q[1], run.E[1]]
    rest = torch.ones(run.npoin, dtype=torch.bool, device="cuda")
    rest[run.lpoin_w.long() - 1] = False
    assert rest.any()
    held[0][rest] = 7.0
    for step in range(3):
        before = [x.clone() for x in held]
        run.step()
        for x, y, b, lv in zip(held, (run.rho, run.q, run.E), before, "rqE"):
            assert x is y[1], (lv, step)
            assert torch.equal(y[0], b) and not torch.equal(x, b), (lv, step)
        assert (held[0][rest] == 7.0).all()


def test_arrays_put_in_the_lists_are_the_levels():
    """A caller may put arrays of its own into run.rho, run.q and run.E."""
    import torch
    from sod2d_amd.solver import TGVRun
    g = make_case(2, 3, periodic=True, lengths=(2 * np.pi,) * 3)
    a, b = (TGVRun(2, geometry=g, parity=False, dt_mode="fixed") for _ in range(2))
    b.q[1] = b.q[1].clone()
    b.E[0] = b.E[0].clone()
    for step in range(3):
        a.step()
        b.step()
        for x, y in zip((a.rho, a.q, a.E), (b.rho, b.q, b.E)):
            assert torch.equal(x[0], y[0]) and torch.equal(x[1], y[1]), step
    a.parity = b.parity = True  # from here on the levels are exchanged
    for step in range(3):
        a.step()
        b.step()
        assert torch.equal(a.E[1], b.E[1]) and torch.equal(a.q[0], b.q[0]), step


@pytest.mark.parametrize("p,precision,lps", [(3, 8, False), (2, 4, False), (4, 8, True)])
def test_captured_steps(p, precision, lps):
    """Two captured steps, the copies of the levels among them, give the bits of eager
    ones on every replay, with the other run's eager work between the replays."""
    import torch
    from sod2d_amd.solver import TGVRun
    g = make_case(p, 3, periodic=True, lengths=(2 * np.pi,) * 3)
    a, b = (TGVRun(p, geometry=g, parity=False, dt_mode="fixed", op_precision=precision, lps=lps)
            for _ in range(2))
    a.step()
    b.step()
    held = b.E[1]
    graph = b.capture()
    for rep in range(4):
        a.step()
        a.step()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert held is b.E[1]
        for x, y in zip((*a.rho, *a.q, *a.E, a.mu_e), (*b.rho, *b.q, *b.E, b.mu_e)):
            assert torch.equal(x, y), rep
    graph.release()


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("precision", [8, 4])
def test_stage_from_level1_is_the_stage_on_a_copy(p, precision):
    import torch
    from sod2d_amd._lib import check, lib
    from sod2d_amd.device import _ptr
    from sod2d_amd.solver import TGVRun
    g = make_case(p, 3, periodic=True, lengths=(2 * np.pi,) * 3)
    run = TGVRun(p, geometry=g, parity=False, dt_mode="fixed", op_precision=precision)
    run.step()
    y1 = [run.rho[1], run.q[1], run.E[1]]
    R = [run.Rmass, run.Rmom, run.Rener]

    def args(lam1, lams, y):
        return (run.ctx.h, p, run.nelem, run.npoin, run.npoin_w, _ptr(run.connec),
                _ptr(run.lpoin_w), precision, _ptr(run.He_op), _ptr(run.gpvol_op),
                _ptr(run.dl_op), *[_ptr(x) for x in run.tabs], _ptr(run.mu_e_op),
                _ptr(run.invMl), C.byref(run.sp), run.dt, lam1, lams, 0.25,
                *[_ptr(x) for x in (*y1, *y, *R)])

    ya = [x.clone() for x in y1]
    check(lib().sodhip_rk_stage_f64(*args(0.0, 1.0, ya)), "rk_stage")
    Ra = [x.clone() for x in R]
    yb = [x.clone() for x in y1]
    w = run.lpoin_w.long() - 1
    for x in yb:  # what the stage overwrites is not read
        x.view(-1, run.npoin)[:, w] = 7.0
    check(lib().sodhip_rk_stage_from_f64(*args(1.0, 0.0, yb), *[_ptr(x) for x in y1]), "from")
    torch.cuda.synchronize()
    for a, b in zip((*ya, *Ra), (*yb, *R)):
        assert torch.equal(a, b)
