"""Position gradients hold their values at every grid size: the rounding of the adjoint's row
pass must not move with the order of its loads.

tests/golden/position_gradients.npz holds 30 atoms and their gradients at each size as this library
gave them (plane wave through SrTiO3, loss sum (I - 1)^2) while the row pass still loaded its
transmission row after its first transform; the same transforms give the same values to the grouping
of FP64 sums."""
import os

import numpy as np
import pytest

import cltem_amd
from cltem_amd import workloads as wl

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "position_gradients.npz")
# FP64 sums over at most 2e5 pixels of equal terms in another grouping; one product of the transforms
# rounded otherwise moves them by 5e-8 and more
TOL = 1e-11


@pytest.mark.parametrize("res", [256, 384, 512, 768, 1024])
def test_gradient_values(res):
    with np.load(GOLDEN) as f:
        x, y, z, Z, want = (f[k] for k in ("x", "y", "z", "Z", f"grad_{res}"))
    w = wl.ctem_srtio3(nx=3, ny=3, nz=2, resolution=res)
    with cltem_amd.Engine(0) as e:
        e.set_geometry(cltem_amd.plan_geometry(cltem_amd.make_scenario(**w["scenario"])))
        e.set_parameterisation(cltem_amd.load_params(w["params"]))
        e.sort_atoms(0, x, y, z, Z)
        e.build_transmission(0)
        e.set_wave_count(1)
        e.set_wave_configs([0])
        e.init_plane_wave()
        I = e.forward_checkpointed(0)
        got = e.adjoint_positions(2.0 * (I - 1.0), len(x))
    assert np.linalg.norm(want) > 0
    assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want)
