"""Waves written through to memory or not, by grid size and number of waves: a wave's result does not
depend on how many run beside it, on either side of the rule."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,few,many", [(256, 1, 40), (384, 2, 30), (512, 3, 20), (768, 17, 18), (768, 1, 24), (1024, 3, 4),
                                          (1024, 1, 9)])
def test_waves_are_the_same_beside_others(engine, res, few, many):
    w = wl.stem_srtio3(nx=3, ny=3, nz=1, resolution=res, pixels=7, window_cells=(1, 2))
    spec = w["specimen"].displaced(0.08, 5, 0)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**w["scenario"]))
    engine.set_geometry(g)
    engine.set_parameterisation(cltem_amd.load_params(w["params"]))
    engine.sort_atoms(0, spec.x, spec.y, spec.z, spec.Z)
    engine.build_transmission(0)
    pos = wl.stem_positions(g)[:many]

    def exits(n):
        engine.set_wave_count(n)
        engine.set_wave_configs([0] * n)
        engine.init_probes(pos[:n], cltem_amd.make_probe(w["cond_ap_mrad"]))
        engine.multislice()
        return [engine.exit_wave(i) for i in (0, few - 1)]

    np.testing.assert_array_equal(exits(few), exits(many))
