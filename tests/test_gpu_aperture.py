"""Scan loops that start from the probes' aperture alone, against probes written over the whole grid:
apertures of one pixel, of a part of the band, at its edge, beyond it and beyond the grid, hard and
tapered, on every grid size and on wave counts either side of the detector tiles' rule."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu

# both sides run the same FP32 passes; only the last column pass may round otherwise, by some 20
# roundings of 2^-24 in the wave and twice that in its intensities: 2.4e-6
TOL = 5e-6


@pytest.mark.parametrize("ap,smooth", [(1e-4, 0.0), (0.1, 0.0), (0.35, 0.1), (0.999, 0.0), (1.2, 0.3), (9.0, 0.0)])
@pytest.mark.parametrize("res,waves", [(256, 3), (256, 17), (384, 3), (512, 9), (768, 2), (1024, 1)])
def test_scan_from_the_aperture_alone(engine, res, waves, ap, smooth):
    w = wl.stem_srtio3(nx=3, ny=3, nz=1, resolution=res, pixels=5, window_cells=(1, 2))
    spec = w["specimen"].displaced(0.08, 5, 0)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**w["scenario"]))
    engine.set_geometry(g)
    engine.set_parameterisation(cltem_amd.load_params(w["params"]))
    engine.sort_atoms(0, spec.x, spec.y, spec.z, spec.Z)
    engine.build_transmission(0)
    band = 1e3 * g.kmax_band * w["scenario"].get("limit_factor", 2.0 / 3.0) * g.wavelength  # in mrad
    probe = cltem_amd.make_probe(ap * band, smooth_mrad=smooth * band, taper=smooth > 0)
    dets = cltem_amd.make_detectors([(0.0, 0.3 * band), (0.2 * band, 0.7 * band), (0.0, 10 * band)])
    pos = wl.stem_positions(g)[:waves]
    engine.set_wave_count(waves)
    engine.set_wave_configs([0] * waves)
    # other waves in the buffers first
    engine.init_probes(pos[::-1].copy(), cltem_amd.make_probe(1.5 * band))
    engine.multislice()
    got = {graph: engine.stem_batch(0, pos, waves, probe, dets, use_graph=graph) for graph in (False, True)}
    np.testing.assert_array_equal(got[False], got[True])
    engine.init_probes(pos, probe)
    engine.multislice()
    want = np.asarray(engine.stem_detect(dets)).reshape(got[True].shape)
    assert np.max(np.abs(got[True] - want)) <= TOL * want.max()
