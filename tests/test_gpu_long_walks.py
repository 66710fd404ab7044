"""The element kernels where a workgroup walks several units: the copies and gathers
of the next units, the two slots of node ids and of viscosities, the records stored one
unit late, and odd p=4 units that start between 16-byte boundaries.

On 256 CUs a workgroup takes three groups of units on these boxes (p=2: from 24,562
elements on, p=3: 12,257, p=4: 6,129), whose odd element counts leave the last group
partly empty.  The boxes are jittered and not periodic: no two elements, and no two
nodes of one, have the same geometry.  Bars as in the tests at the edges of the units
and in the time-loop tests: FP64 operators 1e-13, a step's rho, rho u and E 1e-12, mu_e
1e-10, FP32 operators 2e-5, steps with them 2e-7 (rho, E) and 1e-5 (rho u)."""

import numpy as np
import pytest

import test_gpu_element_units as units
import test_gpu_grad_units as grads
import test_gpu_lps as lps_tests
from helpers import make_case, relerr

pytestmark = pytest.mark.gpu

BOX = {2: (31, 29, 31), 3: (25, 23, 23), 4: (19, 19, 19)}
THREADS = 8  # of the oracle


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("dtype,shift", [("float64", 0), ("float64", 1), ("float32", 0),
                                         ("float32", 1)])
def test_operators(p, dtype, shift):
    units.test_operators_at_unit_edges(p, BOX[p], dtype, shift)


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("shift", [0, 1])
def test_gradient_operators(monkeypatch, p, shift):
    grads.test_gradient_operators_at_unit_edges(monkeypatch, p, BOX[p], shift)


@pytest.mark.parametrize("p", [2, 3, 4])
def test_lps_operators(oracle, p):
    lps_tests.test_full_diff_stab(oracle, p, BOX[p], False, 0.05, True)
    lps_tests.test_comp_tau_and_projection(oracle, p, BOX[p], False, 0.05)


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("box", ["long", (3, 3, 3)])
def test_lps_operators_off_16_byte_boundaries(p, box):
    """Geometry in 16-byte and in 4-byte rows is the same in LDS: the same bits."""
    import torch
    from sod2d_amd import device as D
    g = make_case(p, BOX[p] if box == "long" else box, periodic=False, jitter=0.05,
                  lengths=(1.0, 1.1, 0.9))
    m, T = g.mesh, g.tables
    n, ne = m.npoin, m.nelem
    gen = torch.Generator(device="cuda").manual_seed(p)
    rnd = lambda k, lo, hi: (torch.rand(k, generator=gen, dtype=torch.float64,  # noqa: E731
                                        device="cuda") * (hi - lo) + lo)
    rho, u, Tem, mf = rnd(n, .9, 1.1), rnd(3 * n, -1, 1), rnd(n, .9, 1.1), rnd(n, 1e-3, 2e-3)
    mue, tau = rnd(ne * T.nnode, 0, 1e-2), rnd(ne, .05, .2)
    connec, lw, invMl, dl = (D.to_dev(x) for x in (m.connec, m.lpoin_w, g.invMl, T.dlxigp_ip))
    tabs = [D.to_dev(x) for x in (T.invAtoIJK, T.gmshAtoI, T.gmshAtoJ, T.gmshAtoK)]
    out = []
    for shift in (0, 1):
        He, gv = (units._shifted(D.to_dev(x), shift) for x in (g.He, g.gpvol))
        P = [torch.full((3 * n,), 7.0, dtype=torch.float64, device="cuda") for _ in range(5)]
        R = [torch.full((k * n,), 7.0, dtype=torch.float64, device="cuda") for k in (1, 3, 1)]
        D.full_proj_ijk(ne, n, m.npoin_w, connec, lw, None, He, gv, dl, *tabs, 1004.0, 0.71, rho,
                        u, Tem, None, invMl, *P)
        D.full_diff_stab_ijk(ne, n, connec, None, He, gv, dl, *tabs, 1004.0, 0.71, rho, rho, u,
                             Tem, mf, mue, None, None, *P, tau, *R, initialze=True, fact=-1.0)
        out.append([*P, *R])
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and torch.equal(a, b)


def _runs(oracle, p, box, steps, precision=8, lps=False, parity=True, ctx=None):
    from sod2d_amd.solver import TGVParams, TGVRun
    g = make_case(p, box, periodic=False, jitter=0.05, lengths=(2 * np.pi,) * 3, seed=11)
    tp, to = TGVParams(), oracle.tgv_params()
    ic = oracle.tgv_ic(g.mesh.coord, to)
    kw = dict(sensor_path="live", lps=True) if lps else {}
    run = TGVRun(p, geometry=g, params=tp, initial=ic, parity=parity, op_precision=precision,
                 ctx=ctx, **kw)
    orc = oracle.TGVOracle(p, g, ic, to, parity=parity, cfl=(tp.cfl_conv, tp.cfl_diff),
                           nthreads=THREADS, **kw)
    bars = dict(rho=1e-12, q=1e-12, E=1e-12) if precision == 8 else dict(rho=2e-7, q=1e-5, E=2e-7)
    for step in range(steps):
        run.step()
        orc.step()
        s, w = run.state(), orc.lpoin_w - 1
        for k, bar in bars.items():
            assert relerr(s[k][w], getattr(orc, k)[1][w]) < bar, (k, step)
        if precision == 8:
            assert relerr(s["mu_e"], orc.mu_e) < 1e-10, step


@pytest.mark.parametrize("p,precision,lps", [(2, 8, False), (2, 4, False), (2, 8, True),
                                             (3, 8, False), (3, 4, False), (3, 8, True),
                                             (4, 8, False), (4, 4, False), (4, 8, True)])
def test_time_steps(oracle, p, precision, lps):
    _runs(oracle, p, BOX[p], 2, precision, lps)


@pytest.mark.parametrize("p,box", [(4, 3), (4, (3, 1, 1)), (2, (3, 3, 1)), (3, (5, 1, 1))])
def test_lps_steps_at_unit_edges(oracle, p, box):
    """Odd element counts: a last group of units with one element only."""
    _runs(oracle, p, box, 3, lps=True)


def test_brick_local_steps(oracle, monkeypatch):
    from sod2d_amd.device import Context
    monkeypatch.setenv("SODHIP_STAGE_CLUSTERS", "1")
    ctx = Context(0)
    monkeypatch.delenv("SODHIP_STAGE_CLUSTERS")
    _runs(oracle, 3, BOX[3], 2, ctx=ctx)


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("lps,precision", [(False, 8), (False, 4), (True, 8)])
def test_launch_shapes_agree(p, lps, precision):
    """Units per workgroup (1 block per CU in the setting: sixteen groups) and geometry
    rows change no bit of a step, nor do geometry arrays off 16-byte boundaries."""
    import torch
    from sod2d_amd import autotune
    from sod2d_amd.solver import TGVRun
    g = make_case(p, BOX[p], periodic=False, jitter=0.05, lengths=(2 * np.pi,) * 3, seed=11)
    kw = dict(sensor_path="live", lps=True) if lps else {}
    states = []
    for cfg, shift in (((16, 1, 256), 0), ((1, 1, 256), 0), ((16, 0, 256), 0), ((1, 0, 128), 0),
                       ((16, 1, 256), 1)):
        run = TGVRun(p, geometry=g, dt_mode="fixed", op_precision=precision, **kw)
        if shift:
            run.He_op, run.gpvol_op = (units._shifted(x, 1) for x in (run.He_op, run.gpvol_op))
            if precision == 8:
                run.He, run.gpvol = run.He_op, run.gpvol_op
        was = autotune.get_config(run.ctx)
        autotune.set_config(run.ctx, cfg)
        run.step()
        run.step()
        states.append([x.clone() for x in (run.rho[1], run.q[1], run.E[1], run.mu_e)])
        autotune.set_config(run.ctx, was)
    for s in states[1:]:
        for a, b in zip(states[0], s):
            assert torch.equal(a, b)
