"""The stage's block sizes: one-wave blocks on small 2D meshes (up to 2,048 of
them) and the default above, two elements a block at 3D N = 2.  On both sides
of each line, with full and ragged last blocks, the exact-order stage over
either layout has the bits of volumerhs + facerhs + updatesolution, whose
blocks do not change with the mesh size."""
import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd._lib import EULER, EULER_TE, SWE

from gpu_util import DeviceSetup, dev
from states import smooth_euler_state, smooth_swe_state, smooth_te_state

pytestmark = pytest.mark.gpu


def _setup(eqn, dim, N, sizes):
    L = 1.0 if eqn == SWE else 1000.0
    phys = (P._lib.default_phys(swe_gravity=10.0, delta_nl=1.0) if eqn == SWE
            else P._lib.default_phys(gravity=9.81))
    x = tuple(P.linrange(0.0, L, n + 1) for n in sizes)
    return P.build(eqn, dim, N, x, (True,) + (False,) * (dim - 1), phys=phys)


# 2,048 one-wave blocks: N=4 4,096 elements, N=5 and 6 2,048
@pytest.mark.parametrize("eqn", [EULER, SWE, EULER_TE])
@pytest.mark.parametrize("N,nx,ny", [(4, 64, 64), (4, 65, 63), (4, 241, 17), (5, 64, 32),
                                     (5, 683, 3), (6, 64, 32), (6, 2049, 1)])
def test_2d(cuda, eqn, N, nx, ny):
    check(eqn, 2, N, (nx, ny))


@pytest.mark.parametrize("sizes", [(1, 1, 1), (3, 3, 3), (5, 4, 3)])
def test_3d_order_2(cuda, sizes):
    check(EULER, 3, 2, sizes)


def check(eqn, dim, N, sizes):
    print("case eqn=%d dim=%d N=%d %s" % (eqn, dim, N, sizes), flush=True)
    s = _setup(eqn, dim, N, sizes)
    ds = DeviceSetup(s)
    make = {EULER: smooth_euler_state, SWE: smooth_swe_state, EULER_TE: smooth_te_state}[eqn]
    Q = make(s, seed=4)
    rhs0 = np.asfortranarray(np.random.default_rng(2).standard_normal(Q.shape))
    if eqn == SWE:
        rhs0[:, 3, :] = 0.0
    q, r = dev(Q), dev(rhs0)
    kw = dict(eqn=eqn, phys=s.phys)
    K.volumerhs(dim, N, r, q, ds.vgeo, ds.D, s.nelem, **kw)
    K.facerhs(dim, N, r, q, ds.sgeo, s.nelem, ds.vmapM, ds.vmapP, ds.bndy, vgeo=ds.vgeo, **kw)
    K.updatesolution(dim, N, r, q, ds.vgeo, s.nelem, -0.4, 0.15, 1e-5, eqn=eqn)
    K.check_errors()
    out, rf = torch.full_like(q, float("nan")), dev(rhs0)
    K.stage_fused(dim, N, rf, dev(Q), out, ds.vgeo, ds.sgeo, ds.D, s.nelem, ds.vmapM, ds.vmapP,
                  ds.bndy, -0.4, 0.15, 1e-5, **kw)
    K.check_errors()
    assert torch.equal(out, q) and torch.equal(rf, r)
    if eqn == EULER_TE:  # no prepared form
        return
    prep = K.prepare_geometry(dim, N, ds.vgeo, ds.sgeo, ds.vmapM, ds.vmapP, ds.bndy, s.nelem)
    out.fill_(float("nan"))
    rf = dev(rhs0)
    K.stage_prepared(dim, N, rf, dev(Q), out, prep, ds.D, s.nelem, -0.4, 0.15, 1e-5, **kw)
    K.check_errors()
    assert torch.equal(out, q) and torch.equal(rf, r)
