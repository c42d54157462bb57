"""Sweeps on the band alone: waves whose content starts outside the propagator's band, slices run
in one range or one by one, and limit factors the band does not cover (every column), on every
grid size, against each other and the FP64 oracle."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu

# the waves' bound of the engine's metric: rel-L2 <= 1e-4 against FP64
TOL = 1e-4


@pytest.mark.parametrize("limit", [2.0 / 3.0, 0.5, 0.95])
@pytest.mark.parametrize("res", [256, 384, 512, 768, 1024])
def test_band_sweeps(engine, oracle, res, limit):
    w = wl.stem_srtio3(nx=3, ny=3, nz=1, resolution=res, pixels=2, window_cells=(1, 2))
    scen = dict(w["scenario"], limit_factor=limit)
    spec = w["specimen"].displaced(0.08, 5, 0)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
    og = oracle.geometry(oracle.scenario(**scen))
    p = cltem_amd.load_params(w["params"])
    engine.set_geometry(g)
    engine.set_parameterisation(p)
    engine.sort_atoms(0, spec.x, spec.y, spec.z, spec.Z)
    engine.build_transmission(0)
    # an aperture beyond the band (in mrad: the band limit is kmax_band * limit * wavelength)
    ap = 1.2e3 * g.kmax_band * limit * g.wavelength
    probe = cltem_amd.make_probe(ap)
    pos = wl.stem_positions(g)[:3]
    ns = min(3, g.n_slices)
    engine.set_wave_count(3)
    engine.set_wave_configs([0, 0, 0])

    def exits(ranges):
        engine.init_probes(pos, probe)
        for first, count in ranges:
            engine.multislice(first, count)
        return [engine.exit_wave(i) for i in range(3)], engine.diffraction(2)

    whole, diff = exits([(0, ns)])
    for ranges in ([(s, 1) for s in range(ns)], [(0, 1), (1, ns - 1)]):
        parts, pdiff = exits(ranges)
        for a, b in zip(whole, parts):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(diff, pdiff)
    # nothing outside the propagator's mask (strict <, indices of the shifted pattern)
    k = np.arange(res) - res // 2
    k2 = (k[:, None] ** 2 + k[None, :] ** 2) * g.inverse_scale ** 2
    assert np.all(diff[k2 >= (g.kmax_band * limit) ** 2 * (1 + 1e-12)] <= 1e-10 * diff.max())
    srt = oracle.sort_atoms(og, spec.x, spec.y, spec.z, spec.Z)
    trans = oracle.transmission(og, srt, p.values, p.form, p.i_per_atom, first=0, count=ns)
    P = oracle.propagator(og)
    psi = oracle.fft2(oracle.probe_kspace(og, pos[2][0] - og.sim_x[0], pos[2][1] - og.sim_y[0], cond_ap_mrad=ap),
                      inverse=True)
    for t in trans:
        psi, _ = oracle.slice_step(psi, t, P)
    err = np.linalg.norm(whole[2] - psi) / np.linalg.norm(psi)
    print(f"{res}^2, limit {limit:.3f}: exit wave rel-L2 {err:.2e}")
    assert err <= TOL
