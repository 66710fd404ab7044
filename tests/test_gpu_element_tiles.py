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


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("box", [(1, 1, 1), (5, 3, 1), (4, 2, 2), (17, 1, 1), (11, 3, 1)])
def test_sensor_chunk_edges(p, box):
    """smart_visc_spectral over chunks of 16 elements: the maximum and the filter are
    formed in FP64 (positive weights, fewer than 40 roundings: 1e-13); the FP32
    interface rounds the result once (2^-24: 2e-7)."""
    import torch
    from oracle import oracle as O
    from sod2d_amd import device as D
    from sod2d_amd._lib import check, lib

    g = make_case(p, box, periodic=False, jitter=0.05, lengths=(1.0, 1.1, 0.9))
    m, T = g.mesh, g.tables
    n, ne, nn = m.npoin, m.nelem, T.nnode
    r = np.random.default_rng(40 + p)
    f = dict(Reta=r.normal(0, 1.0, n) * 10.0 ** r.uniform(-2, 4, n), rho=r.uniform(0.9, 1.1, n),
             u=np.asfortranarray(r.normal(0, 0.3, (n, 3))), Tem=r.uniform(0.9, 1.1, n),
             eta=r.normal(size=n), h=g.helem_l, hk=g.helem)
    OT = O.Tables(p)
    up = D.to_dev
    connec, lw, inv = up(m.connec), up(m.lpoin_w), up(T.invAtoIJK)
    prm = D.visc_params(287.0)
    for dt, tol in ((torch.float64, 1e-13), (torch.float32, 2e-7)):
        d = {k: up(v).to(dt) for k, v in f.items()}
        mu, ml = (torch.full((ne * nn,), 7.0, dtype=dt, device="cuda") for _ in range(2))
        if dt == torch.float64:
            D.smart_visc_spectral(ne, n, m.npoin_w, connec, lw, d["Reta"], None, None, None, None,
                                  None, 1.4, d["rho"], d["u"], None, d["Tem"], d["eta"], d["h"],
                                  d["hk"], None, mu, inv, None, None, None, ml, prm)
            o = f
        else:
            ctx = D.Context(0)
            ptr = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
            torch.cuda.synchronize()
            check(lib().sodhip_smart_visc_spectral_f32(
                ctx.h, p, ne, n, m.npoin_w, ptr(connec), ptr(lw), ptr(d["Reta"]), C.c_float(1.4),
                ptr(d["rho"]), ptr(d["u"]), ptr(d["Tem"]), ptr(d["eta"]), ptr(d["h"]),
                ptr(d["hk"]), ptr(inv), C.byref(prm), ptr(mu), ptr(ml)), "smart_visc f32")
            o = {k: np.asfortranarray(np.asarray(v, np.float32).astype(np.float64))
                 for k, v in f.items()}
        torch.cuda.synchronize()
        omu, oml = O.smart_visc_spectral(OT, m.connec, m.lpoin_w, o["Reta"],
                                         float(np.float32(1.4)) if dt == torch.float32 else 1.4,
                                         o["rho"], o["u"], o["Tem"], o["eta"], o["h"], o["hk"],
                                         O.visc_params(287.0), fz((ne, nn)))
        assert relerr(ml.cpu().numpy(), oml.ravel(order="F")) < tol
        assert relerr(mu.cpu().numpy(), omu.ravel(order="F")) < tol


# A block's second and later tiles: 8,785 tiles of 16 and 2,197 of 64 elements over the
# 2,048 blocks of 256 CUs at p=2, 2,179 and 2,110 of 16 at p=3 and p=4, each with a part
# of a tile at the end; and p=4 on either side of the line between the two widths
ROUNDS = [(2, (51, 52, 53)), (3, (33, 32, 33)), (4, (33, 33, 31)), (4, (32, 33, 31))]


@pytest.mark.parametrize("p,box", ROUNDS)
def test_tile_rounds(p, box):
    test_tile_edges(p, box)


@pytest.mark.parametrize("p,box", ROUNDS[:3])
def test_sensor_chunk_rounds(p, box):
    test_sensor_chunk_edges(p, box)
