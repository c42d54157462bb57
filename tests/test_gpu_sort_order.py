"""The order of a bin's atoms after binning is that of the input (a stable sort): full-3D transmission
functions depend on it, since the potential's trapezoid carries a value from one atom of a block row
to the next (transmission_potentials_full_3d_d.cl), and the oracle's reproduce it.  The counting sort,
and the radix sort beyond its bins or its histograms' limit."""
import numpy as np
import pytest

import cltem_amd

pytestmark = pytest.mark.gpu

TOL = 1e-5    # transmission functions against FP64, rel-L2 (the bound of the engine's parity tests)
SEEN = 1e-4   # what another order within the bins moves them by at least


def reversed_bins(srt):
    bs = srt["block_start"]
    idx = np.arange(len(srt["x"]))
    for a, b in zip(bs[:-1], bs[1:]):
        idx[a:b] = idx[a:b][::-1]
    return dict(srt, **{c: srt[c][idx] for c in "xyzZ"})


# atoms, box, share of them in range, share of the box's width and depth that they fill; bins; histogram
# entries in Mi (of 256 atoms each)
@pytest.mark.parametrize("n,box,inside,fill", [
    (257, (12.0, 12.0, 8.0), 1.0, 1.0),             # 128: counting
    (6000, (40.0, 40.0, 16.0), 1.0, 1.0),           # 588: counting
    (2000, (200.0, 200.0, 30.0), 1.0, 0.2),         # 13,851: radix, too many bins
    (300000, (160.0, 160.0, 30.0), 0.01, 0.25)])    # 9,196, 10.3 Mi: radix, too large histograms
def test_order_within_bins(engine, oracle, n, box, inside, fill):
    rng = np.random.default_rng(3)
    pos = rng.uniform(0.0, 1.0, (n, 3)) * np.array(box) * (fill, fill, 1.0)
    pos[rng.uniform(0.0, 1.0, n) >= inside, 2] += 1000.0
    Z = rng.integers(1, 30, n).astype(np.int32)
    x, y, z = (np.ascontiguousarray(pos[:, i]) for i in range(3))
    scen = dict(mode=1, resolution=256, slice_thickness=2.0, struct_min=(0.0, 0.0, 0.0), struct_max=box,
                area=(0.0, box[0], 0.0, box[1]), full3d=1, full3d_integrals=4)
    p = cltem_amd.load_params("kirkland")
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
    og = oracle.geometry(oracle.scenario(**scen))
    srt = oracle.sort_atoms(og, x, y, z, Z)
    engine.set_geometry(g)
    engine.set_parameterisation(p)
    got = engine.sort_atoms(0, x, y, z, Z)
    np.testing.assert_array_equal(got["block_start"], srt["block_start"])
    # the slice above the fullest one: the carried value reaches it from there
    s = int(np.argmax(np.diff(srt["block_start"][:: g.blocks_x * g.blocks_y])[1:]))

    def reference(atoms):
        return oracle.transmission(og, atoms, p.values, p.form, p.i_per_atom, first=s, count=1)[0]

    want, other = reference(srt), reference(reversed_bins(srt))
    assert np.linalg.norm(other - want) >= SEEN * np.linalg.norm(want)
    engine.build_transmission(0, s, 1)
    t = engine.read_transmission(0, s)
    assert np.linalg.norm(t - want) <= TOL * np.linalg.norm(want)
