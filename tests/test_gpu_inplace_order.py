"""The in-place kernels' block order on both sides of its line (210 MB of
arrays, at more than 1,024 workgroups an XCD): volumerhs + facerhs +
updatesolution, and volumerhs + facerhs_update, have the bits of the fused
stage, whose order does not change there."""
import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd._lib import EULER, SWE

from gpu_util import DeviceSetup, dev
from states import smooth_euler_state, smooth_swe_state

pytestmark = pytest.mark.gpu


# bytes an element: 2D N=7 8,448 (24,858 elements), N=1 672 (shallow water: 640); 3D N=3 14,976
@pytest.mark.parametrize("eqn,dim,N,sizes", [(EULER, 2, 7, (137, 61)), (EULER, 2, 7, (24858, 1)),
                                             (EULER, 2, 7, (24859, 1)), (SWE, 2, 1, (365, 363)),
                                             (SWE, 2, 1, (575, 573)), (EULER, 3, 3, (21, 21, 20)),
                                             (EULER, 3, 3, (25, 25, 23))])
def test_bits(cuda, eqn, dim, N, sizes):
    print("case eqn=%d dim=%d N=%d %s" % (eqn, dim, N, sizes), flush=True)
    L = 1.0 if eqn == SWE else 1000.0
    phys = (P._lib.default_phys(swe_gravity=10.0, delta_nl=1.0) if eqn == SWE
            else P._lib.default_phys(gravity=9.81))
    x = tuple(P.linrange(0.0, L, n + 1) for n in sizes)
    s = P.build(eqn, dim, N, x, (True,) + (False,) * (dim - 1), phys=phys)
    ds = DeviceSetup(s)
    Q = (smooth_swe_state if eqn == SWE else smooth_euler_state)(s, seed=4)
    rhs0 = np.asfortranarray(np.random.default_rng(2).standard_normal(Q.shape))
    if eqn == SWE:
        rhs0[:, 3, :] = 0.0
    kw = dict(eqn=eqn, phys=s.phys)
    maps = (s.nelem, ds.vmapM, ds.vmapP, ds.bndy)
    wantr, want = dev(rhs0), torch.full((Q.size,), float("nan"), dtype=torch.float64, device="cuda")
    K.stage_fused(dim, N, wantr, dev(Q), want, ds.vgeo, ds.sgeo, ds.D, *maps, -0.4, 0.15, 1e-5,
                  **kw)
    for _ in range(2):  # both walking directions
        q, r = dev(Q), dev(rhs0)
        K.volumerhs(dim, N, r, q, ds.vgeo, ds.D, s.nelem, **kw)
        r2, out = r.clone(), torch.full_like(want, float("nan"))
        K.facerhs(dim, N, r, q, ds.sgeo, *maps, **kw)
        K.facerhs_update(dim, N, r2, q, out, ds.vgeo, ds.sgeo, *maps, -0.4, 0.15, 1e-5, **kw)
        K.updatesolution(dim, N, r, q, ds.vgeo, s.nelem, -0.4, 0.15, 1e-5, eqn=eqn)
        K.check_errors()
        assert torch.equal(q, want) and torch.equal(r, wantr)
        assert torch.equal(out, want) and torch.equal(r2, wantr)
