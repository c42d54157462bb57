"""Moving frames whose last group of slices is shorter than the others (by one to most of its slices),
with a ragged last batch: frames equal to the parallel field give mse_stem_batch's values."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu


# four slices of these batches' frames fit in 512 MiB: 5 slices go in groups of 3 and 2, 7 of 4 and 3,
# 13 of 4, 4, 4 and 1; three slices of 1024^2 by 20: 5 of 3 and 2, 8 of 3, 3 and 2
@pytest.mark.parametrize("res,batch,dz,slices,full3d", [
    (1024, 16, 3.905 / 2, 5, 0), (512, 64, 1.3, 7, 0), (512, 64, 0.7, 13, 0), (512, 64, 3.905 / 2, 5, 1),
    (1024, 20, 3.905 / 2, 5, 0), (1024, 20, 1.0, 8, 0)])
def test_short_last_group(engine, res, batch, dz, slices, full3d):
    w = wl.stem_srtio3(nx=3, ny=3, nz=1, resolution=res, pixels=10, window_cells=(1, 2))
    scen = dict(w["scenario"], slice_thickness=dz, full3d=full3d, full3d_integrals=4)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
    assert g.n_slices == slices
    spec = w["specimen"].displaced(0.08, 13, 0)
    engine.set_geometry(g)
    engine.set_parameterisation(cltem_amd.load_params(w["params"]))
    engine.sort_atoms(0, spec.x, spec.y, spec.z, spec.Z)
    engine.build_transmission(0)
    n = batch + 2
    pos = wl.stem_positions(g)[:n]
    probe = cltem_amd.make_probe(w["cond_ap_mrad"])
    dets = cltem_amd.make_detectors([(60.0, 200.0), (0.0, 20.0)])
    ref = engine.stem_batch(0, pos, batch, probe, dets)
    frames = np.tile([g.sim_x[0], g.sim_y[0]], (n, 1))
    np.testing.assert_array_equal(engine.stem_batch_frames(0, pos, frames, batch, probe, dets), ref)
