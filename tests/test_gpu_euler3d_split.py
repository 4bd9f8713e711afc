"""The FP64 3D stage has two forms by the number of elements: the split form up
to 2,048 waves (polydeg 1 to 6), the direct form beyond.  rhs! at every polydeg
on both sides of that line, on a curved mesh with walls and on a brick with a
ragged element count, against the oracle (the criterion of
test_gpu_euler3d.py); steps and the resident loop, whose last stage reduces the
wave speeds, against the host loop; and the direct form's two workgroup shapes
at odd element counts beyond the line."""
import numpy as np
import pytest

import trixiatmo_hip as T
from test_gpu_euler3d import check_rhs

pytestmark = pytest.mark.gpu

# trees per face and layers of a shell beyond the line (2,048 / waves per element
# = 512, 512, 409, 227, 128, 186 elements at polydeg 1..6; polydeg 7: always direct)
BEYOND = {1: (8, 2), 2: (8, 2), 3: (9, 1), 4: (7, 1), 5: (5, 1), 6: (6, 1), 7: (2, 1)}
EC = dict(volume_flux="flux_ranocha", surface_flux="flux_ranocha")


def windy(mesh, u0):
    u0 = u0.copy()
    u0[1:4] += 10.0 * np.sin(mesh.node_coordinates / 1e6) * u0[0]
    return u0


@pytest.mark.parametrize("fluxes", [{}, EC], ids=["kg_llf", "ec"])
@pytest.mark.parametrize("beyond", [False, True])
@pytest.mark.parametrize("polydeg", [1, 2, 3, 4, 5, 6, 7])
def test_rhs_on_both_sides_of_the_line(oracle, polydeg, beyond, fluxes):
    trees, layers = BEYOND[polydeg] if beyond else (2, 2)
    mesh, eq, solver, bcs, u0 = T.workloads.shell(trees, layers, polydeg=polydeg, seed=polydeg,
                                                  **fluxes)
    check_rhs(oracle, mesh, eq, solver, bcs, windy(mesh, u0))


@pytest.mark.parametrize("precision", ["fp64", "fp32_geometry"])
@pytest.mark.parametrize("polydeg", [1, 2, 3, 4, 5, 6])
def test_split_form_steps_and_resident_loop(polydeg, precision):
    mesh, eq, solver, bcs, u0 = T.workloads.periodic_cube(trees=3, polydeg=polydeg, seed=4,
                                                          precision=precision)
    print(f"case: E={mesh.n_elements} polydeg {polydeg} {precision}", flush=True)
    semi = T.SemidiscretizationHyperbolic(mesh, eq, solver, bcs)
    semi.set_state(u0)
    t_end = 6.5 * semi.max_dt(0.5)
    a, steps = T.solve(semi, u0, (0.0, t_end), 0.5)
    b, resident = T.solve(semi, u0, (0.0, t_end), 0.5, resident=True, check_every=3)
    assert steps == resident and np.isfinite(a).all()
    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("polydeg,trees", [(3, (9, 7, 7)), (4, (7, 7, 5))])
def test_direct_form_shapes_are_bit_identical(polydeg, trees):
    """one and two elements per workgroup, an odd count beyond the line"""
    mesh = T.P4estMesh(trees, polydeg=polydeg, coordinates_min=(0.0, 0.0, 0.0),
                       coordinates_max=(1.0, 1.2, 0.8))
    eq = T.CompressibleEulerEnergyEquationsWithGravity3D(c_p=1004.0, c_v=717.0, gravity=9.81)
    solver = T.DGSEM(polydeg=polydeg, surface_flux=("flux_lax_friedrichs", "flux_zero"),
                     volume_integral=T.VolumeIntegralFluxDifferencing(("flux_ranocha",
                                                                       "flux_zero")))
    u0 = T.initial_condition_periodic_modes(mesh, eq, 3)
    semi = T.SemidiscretizationHyperbolic(mesh, eq, solver)
    semi.set_state(u0)
    dt = semi.max_dt(0.5)
    got = []
    for v in (0, 1):
        semi.set_kernel_variant(v)
        du = semi.rhs(None, u0)
        semi.set_state(u0)
        semi.step(dt, 3)
        u = semi.get_state()
        semi.set_state(u0)
        semi.set_time(0.0)
        semi.solve_resident(3.5 * dt, 0.5, 2)
        got.append((du, u, semi.get_state()))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("polydeg,trees,one_shape", [(3, (409, 1, 1), True), (3, (410, 1, 1), False),
                                                     (4, (227, 1, 1), True), (4, (228, 1, 1), False)])
def test_autotuner_on_both_sides_of_the_line(polydeg, trees, one_shape):
    """the split form is one kernel for either variant: the tuner chooses 0 and
    reports its one time for both; beyond the line each shape has a time of its
    own"""
    mesh = T.P4estMesh(trees, polydeg=polydeg, coordinates_min=(0.0, 0.0, 0.0),
                       coordinates_max=(float(trees[0]), 1.0, 1.0))
    eq = T.CompressibleEulerEnergyEquationsWithGravity3D(c_p=1004.0, c_v=717.0, gravity=9.81)
    solver = T.DGSEM(polydeg=polydeg, surface_flux=("flux_lax_friedrichs", "flux_zero"),
                     volume_integral=T.VolumeIntegralFluxDifferencing(("flux_ranocha",
                                                                       "flux_zero")))
    semi = T.SemidiscretizationHyperbolic(mesh, eq, solver)
    semi.set_state(T.initial_condition_periodic_modes(mesh, eq, 3))
    runs = [semi.autotune() for _ in range(3)]
    assert all(ms[0] > 0 and ms[1] > 0 for _, ms in runs)
    if one_shape:
        assert all(chosen == 0 and ms[0] == ms[1] for chosen, ms in runs), runs
    else:
        assert any(ms[0] != ms[1] for _, ms in runs), runs
    semi.set_kernel_variant(1)  # accepted on both sides
