"""Every workgroup shape of the covariant stage kernel (node lanes that do all
the work, or split over three sets of waves) gives the same bits, at every
polydeg, for each volume form and both geometry storages: rhs!, steps and the
resident loop, whose last stage reduces the wave speeds.  The element counts
leave a partly filled last workgroup.  The shape a handle starts with is held
to the oracle in test_gpu_swe.py."""
import numpy as np
import pytest

from trixiatmo_hip import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32_geometry"])
@pytest.mark.parametrize("setup", ["isolated_mountain", "geostrophic_balance",
                                   "central"])
@pytest.mark.parametrize("polydeg", [1, 2, 3, 4, 5, 6, 7])
def test_covariant_shapes_are_bit_identical(polydeg, setup, precision):
    print(f"case: polydeg {polydeg} {setup} {precision}", flush=True)
    if setup == "central":
        case = W.covariant_elixir("rossby_haurwitz", cells=3, polydeg=polydeg,
                                  precision=precision,
                                  volume_flux=("flux_central", "flux_nonconservative_ec"),
                                  surface_flux=("flux_lax_friedrichs",
                                                "flux_nonconservative_ec"))
    else:
        case = W.covariant_elixir(setup, cells=3, polydeg=polydeg, precision=precision)
    semi = case.semi()
    rng = np.random.default_rng(polydeg)
    u0 = case.u0() * (1.0 + 0.002 * rng.standard_normal(semi.shape))
    semi.set_state(u0)
    dt = semi.max_dt(0.3)
    first = None
    for v in range(6):
        semi.set_kernel_variant(v)
        semi.set_state(u0)
        semi.set_time(0.0)
        du = semi.rhs(None, u0)
        semi.step(dt, 3)
        steps, t = semi.solve_resident(5.5 * dt, 0.3)
        got = (du, semi.get_state(), steps)
        assert np.isfinite(got[1]).all(), (v, steps, t, np.isfinite(du).all())
        if first is None:
            first = got
        else:
            for a, b in zip(got, first):
                np.testing.assert_array_equal(a, b)
