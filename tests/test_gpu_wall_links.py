"""The one-pass Bouzidi correction where links read each other's slots: cells
with walls on both sides and in both neighbours (all 26 directions of every
listed cell cut, q on both sides of 0.5), so that a link's sources are other
links' destinations and whole lines of links have to share a work entry.

Shapes: entries that end inside a group's neighbourhood (one and three
blocks), and 17 blocks in a row, whose lines of 136 cells give groups of 272
links, longer than one entry's 256.  The oracle corrects from a full copy of
the post-collision populations (bouzidi_kernel.jl:13-92); bar: strict build
bit-identical, flow and thermal populations."""
import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from parity_helpers import compare, run_pair
from test_gpu_boundary_blocks import _box


def _cut(level, every, seed, most=1.0):
    """All directions of every `every`-th cell cut at a random distance.  With
    every cell cut nearer than 0.5, each link reads both of its line's
    neighbours' slots, and a line of m cells is one group of 2 m links."""
    rng = np.random.default_rng(seed)
    cell = np.arange(0, level.n_blocks * 512, every)
    cell = cell[level.obstacle.reshape(-1)[cell] == 0]
    c = cell % 512
    level.bouzidi_cells = np.stack([cell // 512 + 1, c % 8 + 1, (c // 8) % 8 + 1, c // 64 + 1], 1).astype(np.int32)
    q = rng.uniform(0.05, most, (len(cell), 27)).astype(np.float16)
    q[:, 13] = 0
    level.bouzidi_q = q.view(np.uint16)
    level.bouzidi_tri = np.zeros((len(cell), 27), np.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16])
@pytest.mark.parametrize("shape,every", [((1, 1, 1), 1), ((3, 1, 1), 1), ((2, 2, 1), 3), ((17, 1, 1), 1)])
def test_links_through_each_other_strict_bitexact(hip_device, shape, every, storage):
    cfg, _ = cases.tiny_sphere(8, 1, ddf=True)
    cfg = cfg.replace(ramp_steps=2, forces_enabled=False, limiter="none")
    grids, params = _box(*shape)
    if shape[0] == 17:
        grids[0].obstacle[:] = 0
        _cut(grids[0], every, 11, most=0.45)
    else:
        _cut(grids[0], every, 11)
    for wide in (False, True):
        s, o = run_pair(cfg, grids, params, None, steps=2, strict=True, batch=2, storage=storage, amp=0.02,
                        wide_offsets=wide)
        res = compare(s, o, grids, ("f", "rho", "vel", "g", "T"))
        s.close()
        o.close()
        for k, (mx, n, _) in res.items():
            assert mx == 0.0, f"{shape} every {every} wide {wide} {k}: max |diff| {mx} over {n} entries"
