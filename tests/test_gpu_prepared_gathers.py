"""The exact-order prepared 3D stage below N = 6, which gathers early on meshes
of at most one wave a SIMD (1,024 waves): on both sides of that line, in both
walking directions, it has the bits of the reference-array stage."""
import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd._lib import EULER

from gpu_util import DeviceSetup, dev
from states import smooth_euler_state

pytestmark = pytest.mark.gpu


# elements of 1,024 waves: N=1 8,192, N=2 2,048, N=3 1,024, N=4 512, N=5 256
@pytest.mark.parametrize("N,sizes", [(1, (2, 2, 2)), (1, (32, 16, 16)), (1, (8193, 1, 1)),
                                     (2, (16, 16, 8)), (2, (683, 3, 1)), (3, (16, 8, 8)),
                                     (3, (41, 25, 1)), (4, (8, 8, 8)), (4, (27, 19, 1)),
                                     (5, (8, 8, 4)), (5, (257, 1, 1))])
def test_bits(cuda, N, sizes):
    print("case N=%d %s" % (N, sizes), flush=True)
    x = tuple(P.linrange(0.0, 1000.0, n + 1) for n in sizes)
    s = P.build(EULER, 3, N, x, (True, False, False), phys=P._lib.default_phys(gravity=9.81))
    ds = DeviceSetup(s)
    Q = smooth_euler_state(s, seed=4)
    rhs0 = np.asfortranarray(np.random.default_rng(2).standard_normal(Q.shape))
    wr, want = dev(rhs0), torch.empty(Q.size, dtype=torch.float64, device="cuda")
    K.stage_fused(3, N, wr, dev(Q), want, ds.vgeo, ds.sgeo, ds.D, s.nelem, ds.vmapM, ds.vmapP,
                  ds.bndy, -0.4, 0.15, 1e-5, phys=s.phys)
    prep = K.prepare_geometry(3, N, ds.vgeo, ds.sgeo, ds.vmapM, ds.vmapP, ds.bndy, s.nelem)
    two = torch.empty(2, Q.size, dtype=torch.float64, device="cuda")
    for qin, out in ((two[0], two[1]), (two[1], two[0])):
        qin.copy_(dev(Q))
        out.fill_(float("nan"))
        r = dev(rhs0)
        K.stage_prepared(3, N, r, qin, out, prep, ds.D, s.nelem, -0.4, 0.15, 1e-5, phys=s.phys)
        K.check_errors()
        assert torch.equal(out, want) and torch.equal(r, wr)
