"""The per-element reductions and limiters at the edges of their 16-element tiles
(element counts 1, 15, 16, 17, 33), against the oracle: comp_tau, the live-path
sensor, the Ducros limit and the CFL time step.  Maxima are exact and each value
takes fewer than 20 roundings: 1e-13 of the result."""
import ctypes as C

import numpy as np
import pytest

from helpers import fz, make_case, random_state, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("box", [(1, 1, 1), (5, 3, 1), (4, 2, 2), (17, 1, 1), (11, 3, 1)])
def test_tile_edges(p, box):
    import torch
    from oracle import oracle as O
    from sod2d_amd import device as D
    from sod2d_amd._lib import check, lib
    from sod2d_amd.device import _ptr

    g = make_case(p, box, periodic=False, jitter=0.05, lengths=(1.0, 1.1, 0.9))
    m, T = g.mesh, g.tables
    n, ne = m.npoin, m.nelem
    f = random_state(n, ne, T.nnode, seed=5)
    r = np.random.default_rng(2)
    cs = np.sqrt(1.4 * f["pr"] / f["rho"])
    Reta, eta, divU = r.normal(size=n), r.normal(size=n), r.normal(size=n) * g.Ml
    vort = np.asfortranarray(r.normal(size=(n, 3)))
    up = D.to_dev
    connec, lw = up(m.connec), up(m.lpoin_w)
    d = {k: up(f[k]) for k in ("rho", "u", "Tem", "mu_fluid", "mu_e", "mu_sgs")}
    csd, h = up(cs), up(g.helem)

    tau = torch.zeros(ne, dtype=torch.float64, device="cuda")
    D.comp_tau(ne, n, connec, csd, d["u"], h, 0.0, tau)
    assert relerr(tau.cpu().numpy(), O.comp_tau(p, m.connec, cs, f["u"], g.helem)) < 1e-13

    mue = d["mu_e"].clone()
    muel = torch.zeros_like(mue)
    prm = D.visc_params(1.0)
    D.smart_visc_spectral_imex(ne, n, m.npoin_w, connec, lw, up(Reta), None, None, None, None,
                               None, 1.4, d["rho"], d["u"], csd, d["Tem"], up(eta), None, h, None,
                               mue, None, None, None, None, muel, prm)
    omu, oml = fz((ne, T.nnode)), fz((ne, T.nnode))
    omu[...] = f["mu_e"]
    OT = O.Tables(p)
    O.smart_visc_spectral_imex(OT, m.connec, m.lpoin_w, Reta, f["rho"], f["u"], cs, eta, g.helem,
                               O.visc_params(1.0), omu, oml)
    assert relerr(mue.cpu().numpy(), omu.ravel(order="F")) < 1e-13
    assert np.array_equal(muel.cpu().numpy(), f["mu_e"].ravel(order="F"))

    D.ducros_visc_limit(ne, n, m.npoin_w, connec, lw, None, None, None, None, None, None, d["u"],
                        up(divU), up(vort), None, up(g.helem_l), None, up(g.Ml), mue, None, None,
                        None, None, None)
    O.ducros_visc_limit(OT, m.connec, f["u"], divU, vort, g.Ml, g.helem_l, omu, 0.1)
    assert relerr(mue.cpu().numpy(), omu.ravel(order="F")) < 1e-13

    dt = C.c_double()
    ctx = D.default_context()
    check(lib().sodhip_adapt_dt_cfl_f64(
        ctx.h, p, ne, n, _ptr(connec), _ptr(h), _ptr(d["u"]), _ptr(csd), 0.5, 0.4,
        _ptr(d["mu_fluid"]), _ptr(d["mu_sgs"]), _ptr(d["mu_e"]), _ptr(d["rho"]), C.byref(dt)),
        "adapt_dt_cfl")
    ref = O.adapt_dt_cfl(p, m.connec, g.helem, f["u"], cs, 0.5, 0.4, f["mu_fluid"], f["mu_sgs"],
                         f["mu_e"], f["rho"])
    assert abs(dt.value - ref) <= 1e-13 * ref
