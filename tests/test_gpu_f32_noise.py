"""The FP32 drop-in operators on nodal noise, where a field has no mean to remove from
its derivative: their error against the FP64 oracle on the rounded inputs.

Bounds, of the residual's 2-norm, on this box (12 x 13 x 11 elements): what separate FP32
derivatives of each field, summed line by line, leave, measured (convection's mass,
momentum and energy 7.0, 12, 7.2e-8 at every order; viscous momentum 5.9, 6.6, 7.1e-8 at
p = 2, 3, 4), with 4 % for another draw of the noise."""
import numpy as np
import pytest

from helpers import fz, make_case, random_state, relerr

pytestmark = pytest.mark.gpu

CONVECTION = (7.3e-8, 12.6e-8, 7.5e-8)
VISCOUS_MOMENTUM = {2: 6.2e-8, 3: 6.9e-8, 4: 7.4e-8}


@pytest.mark.parametrize("p", [2, 3, 4])
def test_noise_is_as_exact_as_with_separate_derivatives(p):
    import torch
    from oracle import oracle as O
    from sod2d_amd import device as D

    g = make_case(p, (12, 13, 11), periodic=False, jitter=0.03, lengths=(2 * np.pi,) * 3)
    m, T = g.mesh, g.tables
    n = m.npoin
    f = random_state(n, m.nelem, T.nnode, seed=11 + p)
    r = lambda a: np.asfortranarray(np.asarray(a, np.float32).astype(np.float64))  # noqa: E731
    up = lambda a: D.to_dev(a).float()  # noqa: E731
    He, gv, dl, connec = up(g.He), up(g.gpvol), up(T.dlxigp_ip), D.to_dev(m.connec)
    tabs = [D.to_dev(x) for x in (T.invAtoIJK, T.gmshAtoI, T.gmshAtoJ, T.gmshAtoK)]
    d = {k: up(f[k]) for k in ("rho", "u", "q", "pr", "h", "Tem", "mu_fluid", "mu_e", "mu_sgs")}
    Rc, Rd = ([torch.zeros(k * n, dtype=torch.float32, device="cuda") for k in (1, 3, 1)]
              for _ in range(2))
    D.full_convec_ijk(m.nelem, n, connec, None, None, He, gv, dl, None, *tabs, d["u"], d["q"],
                      d["rho"], d["pr"], d["h"], *Rc, initialze=True, fact=-1.0)
    D.full_diffusion_ijk(m.nelem, n, connec, None, He, gv, dl, *tabs, 3.5, 0.71, d["rho"],
                         d["rho"], d["u"], d["Tem"], d["mu_fluid"], d["mu_e"], d["mu_sgs"], None,
                         *Rd, initialze=True, fact=-1.0)
    OT = O.Tables(p)
    OT.dlxigp_ip = r(OT.dlxigp_ip)
    oc, od = ([np.zeros(n), fz((n, 3)), np.zeros(n)] for _ in range(2))
    O.full_convec_ijk(OT, m.connec, r(g.He), r(g.gpvol), r(f["u"]), r(f["q"]), r(f["rho"]),
                      r(f["pr"]), r(f["h"]), *oc, True, -1.0)
    O.full_diffusion_ijk(OT, m.connec, r(g.He), r(g.gpvol), float(np.float32(3.5)),
                         float(np.float32(0.71)), r(f["rho"]), r(f["rho"]), r(f["u"]), r(f["Tem"]),
                         r(f["mu_fluid"]), r(f["mu_e"]), r(f["mu_sgs"]), *od, True, -1.0)
    err = [relerr(a.cpu().numpy(), b.ravel(order="F")) for a, b in zip([*Rc, *Rd], [*oc, *od])]
    for e, bound in zip(err[:3], CONVECTION):
        assert e < bound, err
    assert err[4] < VISCOUS_MOMENTUM[p], err
