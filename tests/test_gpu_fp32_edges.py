"""The FP32 arithmetic at the ends of its range: depths and densities of zero,
subnormal and near the largest numbers, infinite rho*theta.  A dry or empty
node has an infinite wave speed, so the face terms of height and mass are not
finite there (a NaN speed would be dropped by the maximum of the two sides);
subnormal and huge depths give what IEEE divisions give.

Tolerance (huge depths): as for ordinary states, an entry sums at most 60
terms rounded to 2^-24 a few times each: 2e-5 in relative L2."""
import numpy as np
import pytest
import torch

import canary_amd.problems as P
from canary_amd._lib import FP32, SWE
from canary_amd.batch import Batch, Batch32
from canary_amd.perturb import Perturb32
from oracle import oracle as O

from gpu_util import host
from states import rel_l2, small_setup, smooth_swe_state, warped_setup

pytestmark = pytest.mark.gpu


def face_nodes(dim, N):
    ax = np.meshgrid(*[np.arange(N + 1)] * dim, indexing="ij")
    return np.any([(a == 0) | (a == N) for a in ax], axis=0).ravel(order="F")


def register(s, Q, prepared, one_launch=False):
    b = Batch(SWE, 2, prec=FP32, prepared=prepared)
    i = b.add(s, 1e-3, Q=Q)
    b.finalize(single_launch=one_launch)
    b.stage(1.0, 0.0)
    b.check()
    return host(b.solves[i].rhs, Q.shape).astype(np.float64)


@pytest.mark.parametrize("prepared", [False, True])
@pytest.mark.parametrize("N", [1, 4, 7])
def test_dry_element(cuda, N, prepared):
    s = warped_setup(SWE, 2, N, Ne=3, periodic=(True, True), seed=3)
    Q = smooth_swe_state(s, seed=1)
    Q[:, 2, :] = 0.1 + np.abs(Q[:, 2, :])  # a face takes b from its own element
    Q[:, 2:, 0] = 0.0
    Q[:, :2, 0] = 0.25
    r = register(s, Q, prepared)
    assert not np.isfinite(r[face_nodes(2, N), 2, 0]).any()


@pytest.mark.parametrize("prepared", [False, True])
@pytest.mark.parametrize("depth", [1e-38, 1e-39, 3e-42])
def test_subnormal_depth(cuda, depth, prepared):
    s = small_setup(SWE, 2, 3, periodic=(True, False))
    Q = s.zeros_state()
    Q[:, 3, :] = depth
    Q[:, :2, :] = 0.25 * depth
    assert np.isfinite(register(s, Q, prepared)).all()


@pytest.mark.parametrize("prepared", [False, True])
@pytest.mark.parametrize("depth", [2.0 ** -100, 0.9 * 2.0 ** 126, 1.2 * 2.0 ** 126])
def test_depth_far_from_one(cuda, depth, prepared):
    s = small_setup(SWE, 2, 3, periodic=(True, False))
    s.phys.swe_gravity = 0.0
    Q = s.zeros_state()
    Q[:, 3, :] = np.float32(depth)
    rng = np.random.default_rng(5)
    Q[:, :2, :] = np.float32(depth) * rng.uniform(-0.1, 0.1, size=Q[:, :2, :].shape).astype("f4")
    r, want = register(s, Q, prepared), O.rhs_eval(s, Q)
    for k in range(3):
        assert rel_l2(r[:, k, :], want[:, k, :]) <= 2e-5, k


@pytest.mark.parametrize("form", ["compact", "mixed", "batch"])
@pytest.mark.parametrize("what", ["empty", "infinite rho*theta"])
@pytest.mark.parametrize("dim,N", [(2, 4), (3, 2), (3, 4)])
def test_precision_form(cuda, dim, N, what, form):
    s = small_setup(0, dim, N, Ne=2, periodic=(True,) * dim, gravity=0.0)
    Q0 = P.uniform_rest_state(s, 1.25, 1e5)
    rng = np.random.default_rng(N)
    q = np.zeros(Q0.shape, order="F")
    q[:, :dim, :] = rng.uniform(1.0, 2.0, size=q[:, :dim, :].shape)
    q[:, dim, :] = rng.uniform(-0.1, 0.1, size=q[:, dim, :].shape)
    if what == "empty":
        q[:, dim, 0] = -1.25
    Q = np.asfortranarray(Q0 + q)
    if form == "batch":
        b = Batch32(dim)
        i = b.add(s, 1e-3, Q=Q, Q0=Q0)
        b.finalize()
        qd = b.solves[i].Q[0]
    else:
        pf = Perturb32(s, Q0, Q, mixed=form == "mixed")
        qd = pf.q
    if what != "empty":
        qd.view(s.nelem, dim + 2, s.Np)[0, dim + 1] = float("inf")
    if form == "batch":
        b.stage(1.0, 0.0)
        rd = b.solves[i].rhs
    else:
        pf.stage(1.0, 0.0, 1e-3)
        rd = pf.rhs
    torch.cuda.synchronize()
    r = host(rd, Q0.shape)
    assert not np.isfinite(r[face_nodes(dim, N), dim, 0]).any()
    # nothing reaches the elements that do not touch it
    assert np.isfinite(r[~face_nodes(dim, N), dim, :][:, 1:]).all()


@pytest.mark.parametrize("mixed", [False, True])
def test_node_without_volume(cuda, mixed):
    """MJ = 0 at a node (MJI infinite): the update is infinite there, not NaN."""
    s = small_setup(0, 2, 3, Ne=2, periodic=(True, True), gravity=0.0)
    s.vgeo = np.array(s.vgeo, order="F", copy=True)
    n = 5  # inside the element: no face term
    s.vgeo[n, 4, 0], s.vgeo[n, 5, 0] = 0.0, np.inf
    Q0 = P.uniform_rest_state(s, 1.25, 1e5)
    q = np.zeros(Q0.shape, order="F")
    q[:, :2, :] = np.random.default_rng(0).uniform(1.0, 2.0, size=q[:, :2, :].shape)
    pf = Perturb32(s, Q0, np.asfortranarray(Q0 + q), mixed=mixed)
    pf.stage(1.0, 0.5, 1e-3)
    pf.check()
    got = host(pf.q, Q0.shape)
    assert np.isinf(got[n, :2, 0]).all()
    assert np.isfinite(np.delete(got[:, :, 0], n, axis=0)).all() and np.isfinite(got[:, :, 1:]).all()
