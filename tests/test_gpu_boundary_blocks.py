"""Boundary blocks of the stream-collide and thermal kernels, whose pulls take
the mirror slots and the inlet / outlet values inside the interior blocks'
launch: boxes of one level in which a block misses neighbours on one side, on
two opposite sides, on every side at once (one block), or inside the domain (a
hole in level 1, whose sources give w_k, kernel_cumulant.jl:143-159), and a
domain that ends inside a block (the cells past it take the outlet value).

Strict build against the FP32 oracle from the same perturbed state: every
operation is rounded alike, so populations, density, velocity and temperature
are bit-identical."""
from types import SimpleNamespace

import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from openludwig_amd.domain import BlockLevel, build_neighbor_table
from parity_helpers import compare, run_pair


def _box(nbx, nby, nbz, hole=None, nx=None):
    dims = (nbx, nby, nbz)
    coords = np.array([(x, y, z) for x in range(1, nbx + 1) for y in range(1, nby + 1) for z in range(1, nbz + 1)
                       if (x, y, z) != hole], dtype=np.int32)
    pointer = np.zeros(dims, dtype=np.int32, order="F")
    pointer[coords[:, 0] - 1, coords[:, 1] - 1, coords[:, 2] - 1] = np.arange(1, len(coords) + 1)
    rng = np.random.default_rng(3)
    nb = len(coords)
    solid = (rng.random((nb, 512)) < 0.02).astype(np.uint8)
    sponge = np.where(rng.random((nb, 512)) < 0.1, 0.3, 0.0).astype(np.float32)
    level = BlockLevel(level_id=1, dx=1.0, tau=float(np.float32(0.55)), tau_g=float(np.float32(0.6)), coords=coords,
                       neighbor_table=build_neighbor_table(coords, dims), block_pointer=pointer, grid_dims=dims,
                       obstacle=solid, sponge=sponge, wall_dist=np.full((nb, 512), 100.0, np.float32))
    return [level], SimpleNamespace(nx_coarse=nx or 8 * nbx, ny_coarse=8 * nby, nz_coarse=8 * nbz)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16, N.LB_STORAGE_BF16])
@pytest.mark.parametrize("shape,hole,nx", [((1, 1, 1), None, None), ((3, 1, 2), None, None), ((1, 3, 1), None, None),
                                           ((2, 2, 3), (2, 1, 2), None), ((2, 2, 1), None, 12)])
def test_boundary_pull_strict_bitexact(hip_device, shape, hole, nx, storage):
    cfg, _ = cases.tiny_sphere(8, 1, ddf=True)
    cfg = cfg.replace(inlet_turbulence_intensity=np.float32(0.01), ramp_steps=2, boundary_method="none",
                      forces_enabled=False)
    grids, params = _box(*shape, hole=hole, nx=nx)
    for wide in (False, True):
        s, o = run_pair(cfg, grids, params, None, steps=3, strict=True, batch=2, storage=storage, amp=0.02,
                        wide_offsets=wide)
        res = compare(s, o, grids, ("f", "rho", "vel", "g", "T"))
        s.close()
        o.close()
        for k, (mx, n, _) in res.items():
            assert mx == 0.0, f"{shape} {hole} {nx} wide {wide} {k}: max |diff| {mx} over {n} entries"
