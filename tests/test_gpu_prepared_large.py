"""The contracted prepared 2D stage's wider blocks, taken from two million
nodes on: just below that size, at it and with a ragged last block, in both
walking directions, the exact order gives the reference-array stage's bits
and the contracted form stays within 1e-12 of its own reference-array stage
(its products may be fused differently)."""
import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd._lib import EULER, FP64, FP64_FMA, SWE

from gpu_util import DeviceSetup, dev, host
from states import rel_l2, smooth_euler_state, smooth_swe_state

pytestmark = pytest.mark.gpu


# two million nodes: N=2 222,223 elements (471.4^2), N=4 80,000, N=7 31,250
@pytest.mark.parametrize("eqn", [EULER, SWE])
@pytest.mark.parametrize("N,nx,ny", [(2, 471, 473), (4, 320, 250), (4, 319, 250), (7, 177, 177)])
def test_wide_blocks(cuda, eqn, N, nx, ny):
    print("case eqn=%d N=%d %dx%d" % (eqn, N, nx, ny), flush=True)
    L = 1000.0 if eqn == EULER else 1.0
    phys = (P._lib.default_phys(gravity=9.81) if eqn == EULER
            else P._lib.default_phys(swe_gravity=10.0, delta_nl=1.0))
    s = P.build(eqn, 2, N, (P.linrange(0.0, L, nx + 1), P.linrange(0.0, L, ny + 1)),
                (True, False), phys=phys)
    ds = DeviceSetup(s)
    Q = smooth_euler_state(s, seed=2) if eqn == EULER else smooth_swe_state(s, seed=2)
    rhs0 = np.asfortranarray(np.random.default_rng(1).standard_normal(Q.shape))
    if eqn == SWE:
        rhs0[:, 3, :] = 0.0
    prep = K.prepare_geometry(2, N, ds.vgeo, ds.sgeo, ds.vmapM, ds.vmapP, ds.bndy, s.nelem)
    K.check_errors()
    two = torch.empty(2, Q.size, dtype=torch.float64, device="cuda")
    for prec in (FP64, FP64_FMA):
        rw = dev(rhs0)
        want = torch.empty(Q.size, dtype=torch.float64, device="cuda")
        K.stage_fused(2, N, rw, dev(Q), want, ds.vgeo, ds.sgeo, ds.D, s.nelem, ds.vmapM, ds.vmapP,
                      ds.bndy, -0.4, 0.15, 1e-5, eqn=eqn, phys=s.phys, prec=prec)
        for qin, qout in ((two[0], two[1]), (two[1], two[0])):
            qin.copy_(dev(Q))
            qout.fill_(float("nan"))
            r = dev(rhs0)
            K.stage_prepared(2, N, r, qin, qout, prep, ds.D, s.nelem, -0.4, 0.15, 1e-5, eqn=eqn,
                             phys=s.phys, prec=prec)
            K.check_errors()
            if prec == FP64:
                assert torch.equal(qout, want) and torch.equal(r, rw)
            else:
                assert rel_l2(host(qout, Q.shape), host(want, Q.shape)) <= 1e-12
                assert rel_l2(host(r, Q.shape), host(rw, Q.shape)) <= 1e-12
