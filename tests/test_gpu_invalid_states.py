"""States that are not physical reach the wave speeds as numbers that are not
finite, whatever the short quotients and roots of the kernels make of them (an
infinity or a NaN): max_dt refuses them and so does the resident loop, at its
first step or at the one in which they appear."""
import numpy as np
import pytest

import trixiatmo_hip as T
from trixiatmo_hip import workloads as W

pytestmark = pytest.mark.gpu


def make(family):
    if family == "covariant":
        case = W.covariant_elixir("rossby_haurwitz", cells=3, polydeg=3)
        return case.semi(), case.u0()
    if family == "rainy":
        mesh, eq, solver, src, lim, u0, _ = W.rainy_bubble(cells=(8, 4), polydeg=3, seed=3)
        return T.SemidiscretizationRainy(mesh, eq, solver, source_terms=src, stage_limiter=lim), u0
    mesh, eq, solver, bcs, u0 = W.shell(2, 2, polydeg=3, seed=1)
    return T.SemidiscretizationHyperbolic(mesh, eq, solver, bcs), u0


# the variable that is overwritten at one node (with momentum beside it), and its value
@pytest.mark.parametrize("family,variable,value", [
    ("covariant", 0, 0.0), ("covariant", 0, np.inf), ("covariant", 0, -1.0), ("covariant", 1, np.inf),
    ("rainy", 5, np.inf), ("rainy", 8, np.inf), ("rainy", 8, -250.0), ("rainy", 3, np.inf),
    ("euler3d", 0, 0.0), ("euler3d", 0, np.inf), ("euler3d", 4, np.inf), ("euler3d", 4, -1e5)])
def test_refused(family, variable, value):
    print(f"case: {family} variable {variable} = {value}", flush=True)
    semi, u0 = make(family)
    semi.set_state(u0)
    dt = semi.max_dt(0.4)
    u = np.array(u0, order="F")
    at = (slice(None),) + (1,) * (u.ndim - 2) + (5,)
    bad = u[at].copy()
    bad[{"covariant": 1, "rainy": 3, "euler3d": 1}[family]] += 0.3 * np.abs(bad[0])
    bad[variable] = value
    u[at] = bad
    semi.set_state(u)
    semi.set_time(0.0)
    if not (family == "rainy" and variable == 5):  # the energy is not part of the speeds
        with pytest.raises(T.AtmoError, match="NONFINITE"):
            semi.max_dt(0.4)
    with pytest.raises(T.AtmoError, match="NONFINITE"):
        semi.solve_resident(4.0 * dt, 0.4, 2)
