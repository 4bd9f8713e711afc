"""The graph that a handle keeps for its resident loop is taken again only
while the buffers and launch parameters are the ones it was captured with: runs
in pieces on one handle, with a step of five stages in between (which leaves
the state in the other buffer) and with changed options, give the bits of
handles that run one piece each."""
import numpy as np
import pytest

import trixiatmo_hip as T
from trixiatmo_hip import workloads as W

pytestmark = pytest.mark.gpu


def make(family):
    if family == "covariant":
        case = W.covariant_elixir("rossby_haurwitz", cells=3, polydeg=3)
        return case.semi, case.u0()
    if family == "rainy":
        mesh, eq, solver, src, lim, u0, _ = W.rainy_bubble(cells=(8, 4), polydeg=3, seed=3)
        return (lambda: T.SemidiscretizationRainy(mesh, eq, solver, source_terms=src,
                                                  stage_limiter=lim)), u0
    # 48 elements, either shape the split form, or 486 beyond its line
    trees, layers = (9, 1) if family.endswith("direct") else (2, 2)
    mesh, eq, solver, bcs, u0 = W.shell(trees, layers, polydeg=3, seed=1)
    return (lambda: T.SemidiscretizationHyperbolic(mesh, eq, solver, bcs)), u0


@pytest.mark.parametrize("family", ["covariant", "rainy", "euler3d", "euler3d_direct"])
def test_pieces_on_one_handle(family):
    print(f"case: {family}", flush=True)
    build, u0 = make(family)
    one = build()
    one.set_state(u0)
    dt = one.max_dt(0.4)
    u, t = u0, 0.0
    for piece in range(5):
        fresh = build()
        got = []
        for semi in (one, fresh):
            if piece == 1:
                # members of a covariant or 3D handle in another workgroup shape
                if family == "rainy":
                    semi.enable_newton_stats(True)
                else:
                    semi.set_kernel_variant(1)
            if piece == 2 and family == "rainy":
                semi.enable_newton_stats(False)
            semi.set_state(u)
            semi.set_time(t)
            if piece in (2, 4):
                semi.step(0.5 * dt, 1)
            steps, t_reached = semi.solve_resident(t + (2.5 + piece) * dt, 0.4, 3)
            got.append((semi.get_state(), steps, t_reached))
            if piece == 1 and family == "rainy":
                assert semi.newton_stats()["updates"] > 0
        for a, b in zip(*got):
            np.testing.assert_array_equal(a, b)
        assert np.isfinite(got[0][0]).all() and got[0][1][0] > 2
        u, t = got[0][0].reshape(one.shape, order="F"), got[0][2]


@pytest.mark.parametrize("cells,precision", [(1, "fp64"), (9, "fp64"), (9, "fp32_geometry"),
                                             (10, "fp64")])
def test_control_inside_the_first_stage(cells, precision):
    """up to 512 elements the split shapes take the step control into the first
    stage: the same steps to the same bits as with a kernel of its own (the
    plain shapes, and launches one by one), a last step cut short and a wave
    speed that is not a number included"""
    print(f"case: cells {cells} {precision}", flush=True)
    case = W.covariant_elixir("rossby_haurwitz", cells=cells, polydeg=3, precision=precision)
    u0 = case.u0()
    semi = case.semi()
    semi.set_state(u0)
    dt = semi.max_dt(0.4)
    first = None
    for variant, timing in ((0, False), (3, False), (3, True), (4, False), (5, False)):
        semi.enable_timing(timing)
        semi.set_kernel_variant(variant)
        semi.set_state(u0)
        semi.set_time(0.0)
        a = semi.solve_resident(4.5 * dt, 0.4, 4)
        b = semi.solve_resident(6.7 * dt, 0.4, 1)
        got = (semi.get_state(), a[0], a[1], b[0], b[1])
        assert a[0][0] >= 5 and b[1] == 6.7 * dt
        if first is None:
            first = got
        for x, y in zip(got, first):
            np.testing.assert_array_equal(x, y)
    bad = u0.copy()
    bad[0, 0, 0, -1] = np.nan
    for variant in (0, 3):
        semi.enable_timing(False)
        semi.set_kernel_variant(variant)
        semi.set_state(bad)
        semi.set_time(0.0)
        with pytest.raises(T.AtmoError, match="NONFINITE"):
            semi.solve_resident(dt, 0.4)
