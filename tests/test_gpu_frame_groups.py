"""Moving frames whose transmission functions are built in several groups of slices, the last one
ragged, with a ragged last batch: frames equal to the parallel field give mse_stem_batch's values."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,batch,full3d", [(1024, 16, 0), (1024, 9, 0), (512, 64, 0), (512, 48, 1)])
def test_frame_groups(engine, res, batch, full3d):
    w = wl.stem_srtio3(nx=3, ny=3, nz=2, resolution=res, pixels=8, window_cells=(1, 2))
    scen = dict(w["scenario"], full3d=full3d, full3d_integrals=5)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
    spec = w["specimen"].displaced(0.08, 11, 0)
    engine.set_geometry(g)
    engine.set_parameterisation(cltem_amd.load_params(w["params"]))
    engine.sort_atoms(0, spec.x, spec.y, spec.z, spec.Z)
    engine.build_transmission(0)
    n = batch + 3
    pos = wl.stem_positions(g)[np.arange(n) % 64]
    probe = cltem_amd.make_probe(w["cond_ap_mrad"])
    dets = cltem_amd.make_detectors([(60.0, 200.0), (0.0, 20.0)])
    ref = engine.stem_batch(0, pos, batch, probe, dets)
    frames = np.tile([g.sim_x[0], g.sim_y[0]], (n, 1))
    got = engine.stem_batch_frames(0, pos, frames, batch, probe, dets)
    np.testing.assert_array_equal(got, ref)
