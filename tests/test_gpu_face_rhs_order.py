"""facerhs at the 3D orders that read rhs early or late by the number of
workgroups (256 CUs times those that fit a CU's LDS): on both sides of the
line the exact order has the bits of the face terms within the fused stage,
whose form does not change with the size, and the contracted form is within
1e-12 of them."""
import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd._lib import EULER, FP64, FP64_FMA

from gpu_util import DeviceSetup, dev
from states import smooth_euler_state

pytestmark = pytest.mark.gpu


# the last early and the first late element count: N=1 24,576 (8 a workgroup),
# N=2 8,960 (7 a workgroup), N=6 768, N=7 512
@pytest.mark.parametrize("N,sizes", [(1, (32, 32, 24)), (1, (3449, 1, 7)), (1, (24577, 1, 1)),
                                     (2, (32, 28, 10)), (2, (8961, 1, 1)), (6, (12, 8, 8)),
                                     (6, (769, 1, 1)), (7, (8, 8, 8)), (7, (27, 19, 1))])
def test_both_sides_of_the_line(cuda, N, sizes):
    print("case N=%d %s" % (N, sizes), flush=True)
    x = tuple(P.linrange(0.0, 1000.0, n + 1) for n in sizes)
    s = P.build(EULER, 3, N, x, (True, False, False), phys=P._lib.default_phys(gravity=9.81))
    ds = DeviceSetup(s)
    Q = smooth_euler_state(s, seed=4)
    rhs0 = np.asfortranarray(np.random.default_rng(2).standard_normal(Q.shape))
    rv = dev(rhs0)
    K.volumerhs(3, N, rv, dev(Q), ds.vgeo, ds.D, s.nelem, phys=s.phys)
    want, out = dev(rhs0), torch.empty(Q.size, dtype=torch.float64, device="cuda")
    K.stage_fused(3, N, want, dev(Q), out, ds.vgeo, ds.sgeo, ds.D, s.nelem, ds.vmapM, ds.vmapP,
                  ds.bndy, 1.0, 0.0, 1e-5, phys=s.phys)
    for prec in (FP64, FP64_FMA):
        for _ in range(2):  # both walking directions
            r = rv.clone()
            K.facerhs(3, N, r, dev(Q), ds.sgeo, s.nelem, ds.vmapM, ds.vmapP, ds.bndy,
                      phys=s.phys, prec=prec)
            K.check_errors()
            if prec == FP64:
                assert torch.equal(r, want)
            else:
                assert float((r - want).norm()) <= 1e-12 * float(want.norm())
