"""Projected transmission functions from the LDS copy of the tables against those from the global
tables: the same values, for one to seven elements (five fit the copy), small and large pixels, atoms
at every distance from a pixel, empty slices, a tilted beam (global tables both ways)."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("elements", [1, 3, 5, 6, 7])
@pytest.mark.parametrize("res,cells,tilt", [(256, 1, 0.0), (256, 30, 0.0), (384, 6, 0.0), (384, 6, 4.0), (1024, 2, 0.0)])
def test_lds_tables_give_the_same_values(engine, res, cells, tilt, elements):
    w = wl.ctem_srtio3(nx=cells, ny=cells, nz=2, resolution=res)
    scen = dict(w["scenario"], beam_tilt_mrad=tilt)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
    spec = w["specimen"].displaced(0.1, 7, 0)
    z = spec.z.copy()
    z[z < 0.5 * z.max()] = z.min()  # slices without atoms between the planes
    x, y = spec.x.copy(), spec.y.copy()
    x[0], y[0] = g.sim_x[0] + 37 * g.real_scale, g.sim_y[0] + 11 * g.real_scale  # on a pixel
    Z = np.array([8, 38, 22, 6, 14, 79, 92], np.int32)[np.arange(len(x)) % elements]
    engine.set_geometry(g)
    engine.set_parameterisation(cltem_amd.load_params("kirkland"))
    engine.sort_atoms(0, x, y, z, Z)
    got = []
    try:
        for lds in (True, False):
            engine.set_potential_tables(True, lds=lds)
            engine.build_transmission(0)
            got.append([engine.read_transmission(0, s) for s in range(g.n_slices)])
    finally:
        engine.set_potential_tables(True)
    assert any(np.ptp(t.real) > 0 for t in got[0])
    np.testing.assert_array_equal(got[0], got[1])
