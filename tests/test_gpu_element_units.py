"""The element kernels at the edges of their units: element counts that leave
the last unit or group of units partly empty, meshes smaller than one group, and
geometry arrays that do not start on a 16-byte boundary.  FP64 against the oracle,
FP32 against the FP64 oracle on the rounded inputs.

Tolerances: FP64 sums of about 3 (p+1) products per field with relative error
2^-53 each stay below 1e-13 of the residual's 2-norm; FP32 (2^-24) below 2e-5."""
import numpy as np
import pytest

from helpers import fz, make_case, random_state, relerr

pytestmark = pytest.mark.gpu

# element counts 1, 2, 3, 5, 7 (units of two, groups of two and four), 12 and 63
BOXES = [(1, 1, 1), (2, 1, 1), (3, 1, 1), (5, 1, 1), (7, 1, 1), (3, 2, 2), (7, 3, 3)]


def _shifted(x, elems):
    """A device copy of x that starts `elems` values past an allocation's start."""
    import torch
    buf = torch.zeros(x.numel() + elems + 8, dtype=x.dtype, device="cuda")
    out = buf[elems:elems + x.numel()]
    out.copy_(x)
    return out


@pytest.mark.parametrize("p", [2, 3, 4])
@pytest.mark.parametrize("box", BOXES)
@pytest.mark.parametrize("dtype,shift", [("float64", 0), ("float64", 1), ("float32", 0),
                                         ("float32", 1)])
def test_operators_at_unit_edges(p, box, dtype, shift):
    import torch
    from oracle import oracle as O
    from sod2d_amd import device as D

    g = make_case(p, box, periodic=False, jitter=0.05, lengths=(1.0, 1.1, 0.9))
    m, T = g.mesh, g.tables
    f = random_state(m.npoin, m.nelem, T.nnode, seed=3 + p)
    dt = getattr(torch, dtype)

    def up(a):
        t = D.to_dev(a)
        return t.to(dt) if t.is_floating_point() else t

    He, gpvol = _shifted(up(g.He), shift), _shifted(up(g.gpvol), shift)
    dl, connec = up(T.dlxigp_ip), D.to_dev(m.connec)
    tabs = [D.to_dev(x) for x in (T.invAtoIJK, T.gmshAtoI, T.gmshAtoJ, T.gmshAtoK)]
    d = {k: up(f[k]) for k in ("rho", "u", "q", "pr", "h", "Tem", "mu_fluid", "mu_e", "mu_sgs")}
    n = m.npoin

    def out():
        return [torch.full((k * n,), 7.0, dtype=dt, device="cuda") for k in (1, 3, 1)]

    Rc, Rd = out(), out()
    D.full_convec_ijk(m.nelem, n, connec, None, None, He, gpvol, dl, None, *tabs, d["u"], d["q"],
                      d["rho"], d["pr"], d["h"], *Rc, initialze=True, fact=-1.0)
    D.full_diffusion_ijk(m.nelem, n, connec, None, He, gpvol, dl, *tabs, 3.5, 0.71, d["rho"],
                         d["rho"], d["u"], d["Tem"], d["mu_fluid"], d["mu_e"], d["mu_sgs"], None,
                         *Rd, initialze=True, fact=-1.0)

    if dtype == "float32":  # the oracle takes the inputs as the kernels get them
        r = lambda a: np.asfortranarray(np.asarray(a, dtype=np.float32).astype(np.float64))  # noqa: E731
    else:
        r = np.asfortranarray
    OT = O.Tables(p)
    ref = lambda: (np.zeros(n), fz((n, 3)), np.zeros(n))  # noqa: E731
    oc, od = ref(), ref()
    O.full_convec_ijk(OT, m.connec, r(g.He), r(g.gpvol), r(f["u"]), r(f["q"]), r(f["rho"]),
                      r(f["pr"]), r(f["h"]), *oc, True, -1.0)
    O.full_diffusion_ijk(OT, m.connec, r(g.He), r(g.gpvol), 3.5, 0.71, r(f["rho"]), r(f["rho"]),
                         r(f["u"]), r(f["Tem"]), r(f["mu_fluid"]), r(f["mu_e"]), r(f["mu_sgs"]),
                         *od, True, -1.0)
    tol = 1e-13 if dtype == "float64" else 2e-5
    for a, b in zip([*Rc, *Rd], [*oc, *od]):
        assert relerr(a.cpu().numpy(), np.asarray(b).ravel(order="F")) < tol
