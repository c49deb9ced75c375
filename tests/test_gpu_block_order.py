"""The element-block order of the kernels is one to one: every element is
computed once where runs of blocks are dealt to the XCDs (at least 1,024
blocks per XCD), where a piece is left past the last whole round, and in both
walking directions (the stage from Q to Qout and from Qout to Q)."""
import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd._lib import SWE
from oracle import oracle as O

from gpu_util import DeviceSetup, dev, host
from states import smooth_swe_state

pytestmark = pytest.mark.gpu

EPW = 7  # elements per block of the 2D N = 2 kernels


# blocks per XCD: just below the first dealt launch, one whole number of
# rounds, rounds and a ragged rest
@pytest.mark.parametrize("nx,ny", [(239, 239), (256, 224), (256, 235)])
def test_every_block_once(cuda, nx, ny):
    x = (P.linrange(0.0, 1.0, nx + 1), P.linrange(0.0, 1.0, ny + 1))
    s = P.build(SWE, 2, 2, x, (True, False),
                phys=P._lib.default_phys(swe_gravity=10.0, delta_nl=1.0))
    chunk = -(-(-(-s.nelem // EPW)) // 8)
    print("blocks per XCD %d" % chunk, flush=True)
    assert (chunk < 1024, chunk % 64 == 0) == {(239, 239): (True, False), (256, 224): (False, True),
                                              (256, 235): (False, False)}[(nx, ny)]
    ds = DeviceSetup(s)
    Q = smooth_swe_state(s, seed=3)
    rhs0 = np.asfortranarray(np.random.default_rng(4).standard_normal(Q.shape))
    rhs0[:, 3, :] = 0.0  # the bathymetry has no tendency
    Qo, ro = np.asfortranarray(Q.copy()), rhs0.copy(order="F")
    O.volumerhs(s, ro, Qo, nthreads=8)
    O.facerhs(s, ro, Qo, nthreads=8)
    O.updatesolution(s, ro, Qo, -0.4, 0.15, 1e-5, nthreads=8)
    two = torch.empty(2, Q.size, dtype=torch.float64, device="cuda")
    for qin, qout in ((two[0], two[1]), (two[1], two[0])):
        qin.copy_(dev(Q))
        qout.fill_(float("nan"))
        rhs = dev(rhs0)
        K.stage_fused(2, 2, rhs, qin, qout, ds.vgeo, ds.sgeo, ds.D, s.nelem, ds.vmapM, ds.vmapP,
                      ds.bndy, -0.4, 0.15, 1e-5, eqn=SWE, phys=s.phys)
        K.check_errors()
        assert np.array_equal(host(qout, Q.shape), Qo)
        assert np.array_equal(host(rhs, Q.shape), ro)
