"""The device reductions where their walk over the nodes can go wrong: fewer
nodes than lanes, a last turn that is not full, elements larger than a
workgroup, numbers of states without a kernel of their own, no elements.
The energy is within 1e-13 of an exactly rounded sum (64-bit terms summed in
fixed order: at most (turns + 30) roundings of 2^-53), the shallow-water
step has the host's bits."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

import canary_amd.kernels as K
import canary_amd.problems as P
from canary_amd import _lib
from canary_amd._lib import SWE

from gpu_util import dev
from states import small_setup, smooth_swe_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Np,nstate,nelem", [(1, 1, 1), (8, 2, 5), (27, 4, 19420), (512, 5, 1030),
                                             (1000, 3, 700), (600000, 5, 1), (16, 6, 40000)])
def test_energy_over_node_counts(cuda, Np, nstate, nelem):
    nv, imj = 3, 1
    g = torch.Generator(device="cuda").manual_seed(Np)
    Q = torch.randn(nelem, nstate, Np, generator=g, dtype=torch.float64, device="cuda")
    v = torch.rand(nelem, nv, Np, generator=g, dtype=torch.float64, device="cuda")
    work = torch.empty(_lib.REDUCE_WORK, dtype=torch.float64, device="cuda")
    out = torch.empty((), dtype=torch.float64, device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    rc = _lib.lib().canary_l2energysquared_device(Np, nstate, nv, imj, p(Q), p(v), nelem, p(work),
                                                  p(out), P._stream())
    assert rc == 0
    want = math.fsum((v[:, imj:imj + 1] * Q * Q).sum(1).reshape(-1).cpu().numpy())
    assert abs(float(out) - want) <= 1e-13 * want


@pytest.mark.parametrize("N,Ne", [(1, 4), (3, 200), (7, 91)])
def test_step_has_the_hosts_bits(cuda, N, Ne):
    s = small_setup(SWE, 2, N, Ne=Ne)
    Q = np.asfortranarray(smooth_swe_state(s, seed=N))
    got = float(K.cfl(2, N, dev(s.vgeo), dev(Q), s.nelem, eqn=SWE, phys=s.phys))
    assert got == P.cfl(s, Q)


def test_no_elements(cuda):
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    assert float(K.l2energysquared(2, 3, e, e, 0)) == 0.0
    assert float(K.cfl(2, 3, e, e, 0, eqn=SWE)) == np.finfo(np.float64).max
