"""The kernels that the rule on grid size and wave count takes, on an engine of this file's own that no
other test forces variants on: waves equal bit for bit whatever runs beside them, the 4-column
variant against the default one, and the way back from a forced or tuned variant."""
import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def own():
    with cltem_amd.Engine(0) as e:
        yield e


def load(e, res, pixels, nz=1):
    w = wl.stem_srtio3(nx=3, ny=3, nz=nz, resolution=res, pixels=pixels, window_cells=(1, 2))
    spec = w["specimen"].displaced(0.08, 5, 0)
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**w["scenario"]))
    e.set_geometry(g)
    e.set_parameterisation(cltem_amd.load_params(w["params"]))
    e.sort_atoms(0, spec.x, spec.y, spec.z, spec.Z)
    e.build_transmission(0)
    return wl.stem_positions(g), cltem_amd.make_probe(w["cond_ap_mrad"]), cltem_amd.make_detectors([(60.0, 200.0), (0.0, 20.0)])


def exits(e, pos, probe, which):
    e.set_wave_count(len(pos))
    e.set_wave_configs([0] * len(pos))
    e.init_probes(pos, probe)
    e.multislice()
    return np.stack([e.exit_wave(i) for i in which])


# wave counts on either side of the column passes' write-through, of 4- against 8- and 16-column
# tiles, of the persistent column kernel against the lean one and of the plain row kernel against
# the persistent one
@pytest.mark.parametrize("res,few,many", [
    (256, 1, 40), (256, 12, 100), (384, 2, 30), (384, 1, 90), (512, 3, 20), (512, 8, 64), (768, 1, 24),
    (768, 17, 18), (768, 5, 90), (1024, 1, 9), (1024, 3, 4), (1024, 2, 20)])
def test_waves_do_not_depend_on_their_number(own, res, few, many):
    pos, probe, _ = load(own, res, 10)
    which = (0, few - 1)
    np.testing.assert_array_equal(exits(own, pos[:few], probe, which), exits(own, pos[:many], probe, which))


@pytest.mark.parametrize("res", [256, 384, 512, 768, 1024])
def test_four_column_tiles(own, res):
    """The butterflies, twiddles and products of column variant 7; a compiler that fuses others moves
    the waves of a few slices by some 1e-7."""
    pos, probe, _ = load(own, res, 3, nz=2)
    try:
        waves = {}
        for v in (7, 5):
            own.set_kernel_variant(1, v)
            waves[v] = exits(own, pos, probe, range(len(pos)))
    finally:
        own.set_kernel_variant(1, -1)
    assert np.linalg.norm(waves[5] - waves[7]) <= 1e-6 * np.linalg.norm(waves[7])


@pytest.mark.parametrize("res", [384, 512])
def test_back_to_the_rule(own, res):
    pos, probe, dets = load(own, res, 4)
    want = own.stem_batch(0, pos, 16, probe, dets)
    assert np.all(np.isfinite(want)) and np.all(want > 0)
    for forget in (lambda: (own.set_kernel_variant(0, 2), own.set_kernel_variant(1, 6)), lambda: own.autotune(0, 16, reps=1)):
        forget()
        own.stem_batch(0, pos, 16, probe, dets)
        own.set_kernel_variant(0, -1)
        own.set_kernel_variant(1, -1)
        np.testing.assert_array_equal(own.stem_batch(0, pos, 16, probe, dets), want)
    for bad in ((0, -2), (1, -2), (0, 7), (1, 14), (2, -1)):
        with pytest.raises(cltem_amd.MseError):
            own.set_kernel_variant(*bad)
