"""Captured slice loops after the engine's geometry changed under the same buffers: another limit
factor (another band) and another voltage (other probe optics) must not replay the old graph."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("change", [dict(limit_factor=0.5), dict(voltage_kv=80.0)])
@pytest.mark.parametrize("loop", ["stem", "multislice", "group"])
def test_graphs_follow_the_geometry(loop, change):
    w = wl.stem_srtio3(nx=3, ny=3, nz=2, resolution=256, pixels=4, window_cells=(1, 2))
    spec = w["specimen"].displaced(0.08, 3, 0)
    probe = cltem_amd.make_probe(w["cond_ap_mrad"])
    dets = cltem_amd.make_detectors([(60.0, 200.0), (0.0, 20.0)])

    def values(e, scen, graph):
        g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
        e.set_geometry(g)
        e.sort_atoms(0, spec.x, spec.y, spec.z, spec.Z)
        e.build_transmission(0)
        pos = wl.stem_positions(g)[:4]
        if loop == "stem":
            return e.stem_batch(0, pos, 4, probe, dets, use_graph=graph)
        e.set_wave_count(4)
        e.set_wave_configs([0] * 4)
        e.init_probes(pos, probe)
        if loop == "group" and graph:
            groups.setdefault("g", cltem_amd.EngineGroup([e])).multislice()
        else:
            e.multislice(graph=graph)
        return e.stem_detect(dets)

    groups = {}
    with cltem_amd.Engine(0) as a, cltem_amd.Engine(0) as b:
        for e in (a, b):
            e.set_parameterisation(cltem_amd.load_params(w["params"]))
        for scen in (w["scenario"], dict(w["scenario"], **change), w["scenario"]):
            np.testing.assert_array_equal(values(a, scen, True), values(b, scen, False))
        if groups:
            groups["g"].close()
