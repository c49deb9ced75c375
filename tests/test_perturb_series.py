"""The precision form's pressure series: kappa binomials over |x| <= 1/8.

The polynomial itself, in 64 bits, is within 3e-9 of expm1(kappa log1p(x)) for
every kappa of [1, 2] (its first left-out term is below 0.006 |x|^7).

On the GPU, at the edge of the range and at rest, the momentum register holds
gradients of P' alone.  Roundings of 2^-24 = 6e-8 on the way: background
rho*theta and P0, quotient, coefficients, series, product, 4 in all; metric
terms, MJ, their products and D, 2.5; at most 30 summands, rounded
independently, 2.7; normal, sMJ and the face sums, 2.  Together 11.2, 7e-7 in
relative L2.  Without its last three terms the series would be off by 1.2e-6
to 2e-6."""
import numpy as np
import pytest

import canary_amd.problems as P

from states import rel_l2, small_setup


@pytest.mark.parametrize("kappa", [1.0, 1.1, 1.4, 1.5, 5.0 / 3, 1.9, 2.0])
def test_truncation(kappa):
    x = np.concatenate([np.linspace(-0.125, 0.125, 4001), [1e-6, -1e-6]])
    x = x[x != 0]
    c, b = [], kappa
    for i in range(7):
        c.append(b)
        b = b * (kappa - (i + 1)) / (i + 2)
    a = np.zeros_like(x)
    for v in reversed(c):
        a = a * x + v
    want = np.expm1(kappa * np.log1p(x))
    assert np.max(np.abs(x * a - want) / np.abs(want)) <= 3e-9


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("dim,N,Ne", [(3, 2, 3), (3, 4, 2), (3, 7, 2), (2, 4, 4), (2, 7, 3)])
def test_edge_of_the_range(cuda, dim, N, Ne, mixed):
    from canary_amd.perturb import Perturb32
    from gpu_util import host
    from oracle import oracle as O
    print("case dim=%d N=%d mixed=%s" % (dim, N, mixed), flush=True)
    s = small_setup(0, dim, N, Ne=Ne, gravity=0.0)
    s.phys.c_p = 1.4 * s.phys.c_v
    Q0 = P.uniform_rest_state(s, 1.25, 1e5)
    rng = np.random.default_rng(N)
    q = np.zeros(Q0.shape, order="F")
    size = rng.uniform(0.11, 0.1249, size=q[:, dim + 1, :].shape)
    q[:, dim + 1, :] = Q0[:, dim + 1, :] * size * rng.choice([-1.0, 1.0], size=size.shape)
    pf = Perturb32(s, Q0, np.asfortranarray(Q0 + q), mixed=mixed)
    Q = np.asfortranarray(Q0 + host(pf.q, Q0.shape).astype(np.float64))
    pf.stage(1.0, 0.0, 1e-3)
    pf.check()
    want, got = O.rhs_eval(s, Q), host(pf.rhs, Q0.shape).astype(np.float64)
    for k in range(dim):
        assert rel_l2(got[:, k, :], want[:, k, :]) <= 7e-7, k
