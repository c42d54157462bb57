"""Position gradients of projected potentials on small and large pixels, up to the grid's 64 pixel
groups across and with atoms at its edges: the untilted metric against the tilted one at a tilt far
below the rounding."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu

# each side is one FP32 evaluation within 1e-5 of FP64 (rel-L2, exit wave and adjoint states)
TOL = 4e-5


@pytest.mark.parametrize("tables", [True, False])
@pytest.mark.parametrize("res,cells", [(256, 1), (256, 12), (512, 3), (1024, 2), (1024, 16)])
def test_untilted_metric_is_the_tilted_one(engine, res, cells, tables):
    w = wl.ctem_srtio3(nx=cells, ny=cells, nz=2, resolution=res)
    spec = w["specimen"].displaced(0.1, 3, 0)
    keep = np.argsort(spec.x + spec.y)[np.linspace(0, len(spec.x) - 1, min(60, len(spec.x))).astype(int)]
    x, y, z, Z = (np.ascontiguousarray(v[keep]) for v in (spec.x, spec.y, spec.z, spec.Z))
    grads = []
    try:
        for tilt in (0.0, 1e-9):
            engine.set_geometry(cltem_amd.plan_geometry(cltem_amd.make_scenario(**dict(w["scenario"], beam_tilt_mrad=tilt,
                                                                                         beam_azimuth=0.4))))
            engine.set_parameterisation(cltem_amd.load_params(w["params"]))
            engine.set_potential_tables(tables)
            engine.sort_atoms(0, x, y, z, Z)
            engine.build_transmission(0)
            engine.set_wave_count(1)
            engine.set_wave_configs([0])
            engine.init_plane_wave()
            I = engine.forward_checkpointed(0)
            grads.append(engine.adjoint_positions(2.0 * (I - 1.0), len(x)))
    finally:
        engine.set_potential_tables(True)
    assert np.linalg.norm(grads[1]) > 0
    assert np.linalg.norm(grads[0] - grads[1]) <= TOL * np.linalg.norm(grads[1])
