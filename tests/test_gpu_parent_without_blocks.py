"""A refined level above a level that holds no block: every interpolation corner
is missing, so the ghost cells take the rest state (rest weights, density and
temperature 1, velocity 0; physics_interpolation.jl:85-96).  The parent's
velocity buffer holds one value, so nothing may be read from it in place of a
missing corner.

Strict build against the FP32 oracle, flow and thermal populations:
bit-identical."""
import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from parity_helpers import compare, run_pair
from test_gpu_ghost_groups import _ragged


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16])
@pytest.mark.parametrize("temporal", [True, False])
def test_parent_without_blocks_strict_bitexact(hip_device, temporal, storage):
    cfg, _ = cases.tiny_sphere(8, 1, ddf=True)
    cfg = cfg.replace(ramp_steps=2, forces_enabled=False, temporal_interpolation=temporal)
    grids, params = _ragged((2, 2, 2), 0.4, 7)
    grids = grids[:2]
    parent = grids[0]
    parent.coords = parent.coords[:0]
    parent.neighbor_table = parent.neighbor_table[:0]
    parent.block_pointer = np.zeros_like(parent.block_pointer)
    parent.obstacle, parent.sponge, parent.wall_dist = parent.obstacle[:0], parent.sponge[:0], parent.wall_dist[:0]
    s, o = run_pair(cfg, grids, params, None, steps=3, strict=True, perturb=False, batch=2, storage=storage)
    res = compare(s, o, grids[1:], ("f", "rho", "vel", "g", "T"))
    s.close()
    o.close()
    for k, (mx, n, _) in res.items():
        assert mx == 0.0, f"{k}: max |diff| {mx} over {n} entries"
