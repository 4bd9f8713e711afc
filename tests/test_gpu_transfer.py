"""States of 8 MiB and more come to the host through pinned slots and several
threads: sizes around the threshold and around whole chunks of 2 MiB come back
as they went in, also when two handles are read from two threads at once (one
then finds the slots taken) and after every handle has gone."""
import gc
import threading

import numpy as np
import pytest

import trixiatmo_hip as T

pytestmark = pytest.mark.gpu


def rainy(cells):
    """a handle whose state holds 9 * 4 * cells doubles"""
    mesh = T.meshes.StructuredMesh2D((cells, 1), (0.0, 0.0), (1.0, 1.0), polydeg=1)
    solver = T.DGSEM(polydeg=1, surface_flux="flux_lax_friedrichs",
                     volume_integral=T.VolumeIntegralFluxDifferencing("flux_ec_rain"))
    return T.SemidiscretizationRainy(mesh, T.equations.CompressibleRainyEulerEquations2D(), solver)


def fill(semi, seed):
    u = np.random.default_rng(seed).standard_normal(int(np.prod(semi.shape)))
    semi.set_state(u)
    return u


# 288 bytes a cell: 8 MiB lies between 29,127 and 29,128 cells, a multiple of
# 2 MiB at 65,536 cells (18 MiB)
@pytest.mark.parametrize("cells", [29127, 29128, 65535, 65536, 65537, 131072])
def test_states_come_back(cells):
    print(f"case: {cells} cells", flush=True)
    semi = rainy(cells)
    u = fill(semi, cells)
    np.testing.assert_array_equal(semi.get_state(), u)
    np.testing.assert_array_equal(semi.get_state(), u)


def test_two_threads_and_no_handle_left():
    semis = [rainy(c) for c in (60000, 70001)]
    states = [fill(s, k) for k, s in enumerate(semis)]
    wrong = []

    def read(k):
        for _ in range(5):
            if not np.array_equal(semis[k].get_state(), states[k]):
                wrong.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    semis.clear()
    gc.collect()
    semi = rainy(65536)
    u = fill(semi, 9)
    np.testing.assert_array_equal(semi.get_state(), u)
