"""The 3D reductions at every polydeg, where the lanes of a workgroup (n^3
rounded up to waves: 384 at polydeg 6) need not be a power of two: max_dt finds
the fastest node wherever it lies in its element, and the integrals count every
node, against the oracle.

Tolerances: the integrals sum at most 4,096 terms of one sign, one after the
other in the oracle (4,096 x 1.1e-16 = 4.5e-13) plus a few units per term, held
to 1e-12; a step size is the reciprocal of three sums of three products and one
square root over metric terms that are themselves sums of at most 16 products,
held to 1e-13.  A node left out changes either by far more."""
import numpy as np
import pytest

import trixiatmo_hip as T
from oracle_lib import params_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("polydeg", [1, 2, 3, 4, 5, 6, 7])
def test_reductions_take_every_node(oracle, polydeg):
    print(f"case: polydeg {polydeg}", flush=True)
    mesh, eq, solver, bcs, u0 = T.workloads.periodic_cube(trees=2, polydeg=polydeg, seed=1)
    semi = T.SemidiscretizationHyperbolic(mesh, eq, solver, bcs)
    p = params_for((mesh, eq, solver, 0.0))
    rng = np.random.default_rng(polydeg)
    shape = u0.shape[1:]
    rho, prs = rng.uniform(1.0, 1.5, shape), rng.uniform(4.0, 5.0, shape)
    v = rng.uniform(0.1, 0.5, (3,) + shape)
    u = np.stack([rho, *(rho * v), prs / (eq.c_p / eq.c_v - 1.0) + 0.5 * rho * (v ** 2).sum(0),
                  rng.uniform(1.0, 2.0, shape)])
    semi.set_state(u)
    got = semi.integrals(fresh_rhs=False)
    ref = oracle.integrals(p, mesh, u)
    rows = [0, 1, 3, 4, 5, 6, 7, 8]
    np.testing.assert_allclose(got[rows], ref[rows], rtol=1e-12)
    n3 = (polydeg + 1) ** 3
    flat = u.reshape(6, n3, -1, order="F")
    for node in {0, n3 - 1, n3 // 2, *rng.integers(0, n3, 12)}:
        fast = flat.copy()
        e = int(rng.integers(0, flat.shape[2]))
        fast[1, node, e] += 40.0 * fast[0, node, e]
        fast[4, node, e] += 0.5 * fast[1, node, e] ** 2 / fast[0, node, e]
        fast = fast.reshape(u.shape, order="F")
        semi.set_state(fast)
        dt, dt_ref = semi.max_dt(0.5), 0.5 * oracle.max_dt(p, mesh, fast)
        assert abs(dt / dt_ref - 1) < 1e-13, (node, e, dt, dt_ref)
