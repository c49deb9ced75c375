"""The contracted prepared 2D stage's 256-lane blocks at N=3 (16 elements) and
N=5 (7), from two million nodes on (125,000 and 55,556 elements) with a ragged
last block and just below: within 1e-12 of the exact order in relative L2,
which has the reference-array stage's bits."""
import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd._lib import EULER, FP64, FP64_FMA, SWE

from gpu_util import DeviceSetup, dev
from states import smooth_euler_state, smooth_swe_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eqn,N,nx,ny", [(EULER, 3, 353, 355), (EULER, 5, 236, 236),
                                         (SWE, 3, 357, 351), (SWE, 5, 236, 235)])
def test_against_the_exact_order(cuda, eqn, N, nx, ny):
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
    wr, want = dev(rhs0), torch.empty(Q.size, dtype=torch.float64, device="cuda")
    K.stage_fused(2, N, wr, dev(Q), want, ds.vgeo, ds.sgeo, ds.D, s.nelem, ds.vmapM, ds.vmapP,
                  ds.bndy, -0.4, 0.15, 1e-5, eqn=eqn, phys=s.phys)
    for prec in (FP64, FP64_FMA):
        r, out = dev(rhs0), torch.full_like(want, float("nan"))
        K.stage_prepared(2, N, r, dev(Q), out, prep, ds.D, s.nelem, -0.4, 0.15, 1e-5, eqn=eqn,
                         phys=s.phys, prec=prec)
        K.check_errors()
        if prec == FP64:
            assert torch.equal(out, want) and torch.equal(r, wr)
        else:
            assert float((out - want).norm()) <= 1e-12 * float(want.norm())
            assert float((r - wr).norm()) <= 1e-12 * float(wr.norm())
