"""Binning over the range of atom and bin counts: both sorts, atoms out of range, single bins,
block remainders; bins, their starts and the order within a bin against the oracle's stable sort."""
import numpy as np
import pytest

import cltem_amd

pytestmark = pytest.mark.gpu


# atoms, box, slice thickness: counting sort up to 12,287 bins, radix sort beyond (and for
# histograms over 8 Mi entries)
@pytest.mark.parametrize("n,box,dz", [
    (1, (10.0, 10.0, 4.0), 2.0), (255, (10.0, 10.0, 4.0), 100.0), (256, (30.0, 10.0, 40.0), 1.0),
    (257, (12.0, 40.0, 5.0), 0.5), (5000, (60.0, 60.0, 60.0), 1.0), (70001, (40.0, 40.0, 80.0), 1.0),
    (3000, (200.0, 200.0, 30.0), 2.0), (3000, (200.0, 200.0, 60.0), 1.5), (300000, (90.0, 90.0, 90.0), 1.0)])
def test_sort_ranges(engine, oracle, n, box, dz):
    rng = np.random.default_rng(n)
    p = cltem_amd.load_params("kirkland")
    pos = rng.uniform(-12.0, np.array(box) + 12.0, (n, 3))
    Z = rng.integers(1, 30, n).astype(np.int32)
    scen = dict(mode=1, resolution=256, slice_thickness=dz, struct_min=(0.0, 0.0, 0.0), struct_max=box,
                area=(0.0, box[0], 0.0, box[1]))
    g = cltem_amd.plan_geometry(cltem_amd.make_scenario(**scen))
    og = oracle.geometry(oracle.scenario(**scen))
    engine.set_geometry(g)
    engine.set_parameterisation(p)
    x, y, z = (np.ascontiguousarray(pos[:, i]) for i in range(3))
    got = engine.sort_atoms(0, x, y, z, Z)
    ref = oracle.sort_atoms(og, x, y, z, Z)
    assert got["n_in_range"] == ref["n_in_range"]
    np.testing.assert_array_equal(got["block_start"], ref["block_start"])
    keep = got["block_ids"] >= 0
    np.testing.assert_array_equal(got["block_ids"][keep], ref["block_ids"])
    np.testing.assert_array_equal(got["z_ids"][keep], ref["z_ids"])
    # the order within a bin shows in nothing but the sums' rounding: two sorts of the same atoms
    # give the same transmission functions, and the oracle's order the oracle's values
    if n <= 5000 and g.n_slices <= 200:
        s = int(np.argmax(np.diff(ref["block_start"][:: g.blocks_x * g.blocks_y])))
        engine.build_transmission(0, s, 1)
        t = engine.read_transmission(0, s)
        want = oracle.transmission(og, ref, p.values, p.form, p.i_per_atom, first=s, count=1)[0]
        assert np.linalg.norm(t - want) <= 1e-5 * np.linalg.norm(want)
