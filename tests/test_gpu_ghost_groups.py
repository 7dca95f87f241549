"""The coarse-to-fine ghost fill on ragged refinements: random sets of refined
blocks (faces, edges, lone corners, concave notches, blocks at the domain's low
and high faces), and a third level over a second one with holes, so that
interpolation corners lie in parent blocks that do not exist
(physics_interpolation.jl:89-96).  Dense sets fill work-groups up to their limit
of pairs, sparse ones up to their limits of groups and ghost blocks.

Strict build against the FP32 oracle (which interpolates per cell and
direction), flow and thermal populations: bit-identical."""
from types import SimpleNamespace

import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from openludwig_amd.domain import BlockLevel, build_neighbor_table
from parity_helpers import compare, run_pair


def _level(level_id, active, tau, rng):
    coords = (np.argwhere(active) + 1).astype(np.int32)
    dims = active.shape
    nb = len(coords)
    pointer = np.zeros(tuple(int(v) for v in coords.max(axis=0)), dtype=np.int32, order="F")
    pointer[coords[:, 0] - 1, coords[:, 1] - 1, coords[:, 2] - 1] = np.arange(1, nb + 1)
    return BlockLevel(level_id=level_id, dx=1.0 / 2 ** (level_id - 1), tau=float(np.float32(tau)),
                      tau_g=float(np.float32(0.5 + 1.4 * (tau - 0.5))), coords=coords,
                      neighbor_table=build_neighbor_table(coords, dims), block_pointer=pointer, grid_dims=dims,
                      obstacle=(rng.random((nb, 512)) < 0.01).astype(np.uint8),
                      sponge=np.zeros((nb, 512), np.float32), wall_dist=np.full((nb, 512), 100.0, np.float32))


def _ragged(shape, density, seed):
    rng = np.random.default_rng(seed)
    levels = [_level(1, np.ones(shape, dtype=bool), 0.53, rng)]
    for lvl, tau in ((2, 0.56), (3, 0.62)):
        parent = np.zeros(tuple(s * 2 ** (lvl - 2) for s in shape), dtype=bool)
        c = levels[-1].coords
        parent[c[:, 0] - 1, c[:, 1] - 1, c[:, 2] - 1] = True
        child = np.repeat(np.repeat(np.repeat(parent, 2, 0), 2, 1), 2, 2)
        levels.append(_level(lvl, child & (rng.random(child.shape) < (density if lvl == 2 else 0.5 * density)), tau, rng))
    return levels, SimpleNamespace(nx_coarse=8 * shape[0], ny_coarse=8 * shape[1], nz_coarse=8 * shape[2])


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16])
@pytest.mark.parametrize("shape,density,temporal", [((2, 2, 2), 0.9, True), ((3, 2, 2), 0.4, True),
                                                    ((3, 3, 2), 0.08, True), ((2, 2, 2), 0.5, False)])
def test_ragged_refinement_strict_bitexact(hip_device, shape, density, temporal, storage):
    cfg, _ = cases.tiny_sphere(8, 1, ddf=True)
    cfg = cfg.replace(ramp_steps=2, forces_enabled=False, temporal_interpolation=temporal)
    grids, params = _ragged(shape, density, 7)
    s, o = run_pair(cfg, grids, params, None, steps=3, strict=True, batch=2, storage=storage, amp=0.02)
    res = compare(s, o, grids, ("f", "rho", "vel", "g", "T"))
    s.close()
    o.close()
    for k, (mx, n, _) in res.items():
        assert mx == 0.0, f"{shape} density {density} {k}: max |diff| {mx} over {n} entries"
