"""Projected transmission functions where a wave's pixels lie all, partly or not at all within an
atom's 8 Angstrom, and at its very core: small and large pixels, tabulated and direct, tilted and
not, against the FP64 oracle."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu

TOL = 1e-5  # transmission functions against FP64, rel-L2 (the bound of the engine's parity tests)


@pytest.mark.parametrize("params", ["kirkland", "peng", "lobato"])
@pytest.mark.parametrize("res,cells,tilt", [(256, 3, 0.0), (256, 14, 0.0), (384, 6, 4.0), (512, 2, 0.0), (1024, 2, 0.0)])
def test_projected_slices(engine, oracle, res, cells, tilt, params):
    w = wl.ctem_srtio3(nx=cells, ny=cells, nz=1, resolution=res, params=params)
    scen = dict(w["scenario"], beam_tilt_mrad=tilt, beam_azimuth=0.4)
    spec = w["specimen"].displaced(0.1, 7, 0)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
    og = oracle.geometry(oracle.scenario(**scen))
    p = cltem_amd.load_params(params)
    # one atom exactly on a pixel, where the distance is clamped to a quarter pixel
    x = np.append(spec.x, g.sim_x[0] + 37 * g.real_scale)
    y = np.append(spec.y, g.sim_y[0] + (res - 41) * g.real_scale)
    z = np.append(spec.z, spec.z[0])
    Z = np.append(spec.Z, np.int32(38))
    engine.set_geometry(g)
    engine.set_parameterisation(p)
    engine.sort_atoms(0, x, y, z, Z)
    engine.build_transmission(0)
    srt = oracle.sort_atoms(og, x, y, z, Z)
    counts = np.diff(srt["block_start"][:: g.blocks_x * g.blocks_y])
    s = int(np.argmax(counts))
    ref = oracle.transmission(og, srt, p.values, p.form, p.i_per_atom, first=s, count=1)[0]
    got = engine.read_transmission(0, s)
    err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    print(f"{params} {res}^2, {cells} cells, tilt {tilt}: {counts[s]} atoms, rel-L2 {err:.2e}")
    assert err <= TOL
