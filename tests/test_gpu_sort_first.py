"""Binning before a parameterisation is set: the transmission functions are those of the other order,
and atomic numbers that the parameterisation lacks are refused when potentials are asked for."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("full3d", [0, 1])
def test_sort_before_parameterisation(full3d):
    w = wl.ctem_srtio3(nx=3, ny=3, nz=2, resolution=256)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**dict(w["scenario"], full3d=full3d, full3d_integrals=4)))
    p = cltem_amd.load_params("kirkland")
    s = w["specimen"]

    def functions(sort_first):
        with cltem_amd.Engine(0) as e:
            e.set_geometry(g)
            if not sort_first:
                e.set_parameterisation(p)
            e.sort_atoms(0, s.x, s.y, s.z, s.Z)
            if sort_first:
                e.set_parameterisation(p)
            e.build_transmission(0)
            return np.stack([e.read_transmission(0, k) for k in range(g.n_slices)])

    np.testing.assert_array_equal(functions(True), functions(False))


@pytest.mark.parametrize("Z", [-1, 0, 200, 100000])
def test_unknown_elements_are_refused(Z):
    w = wl.ctem_srtio3(nx=3, ny=3, nz=2, resolution=256)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**w["scenario"]))
    s = w["specimen"]
    numbers = s.Z.copy()
    numbers[5] = Z
    with cltem_amd.Engine(0) as e:
        e.set_geometry(g)
        e.sort_atoms(0, s.x, s.y, s.z, numbers)
        e.set_parameterisation(cltem_amd.load_params("kirkland"))
        with pytest.raises(cltem_amd.MseError):
            e.build_transmission(0)
        e.sort_atoms(0, s.x, s.y, s.z, s.Z)
        e.build_transmission(0)
        assert np.all(np.isfinite(e.read_transmission(0, 0)))
