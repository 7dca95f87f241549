"""Boundary cells that the caller lists more than once.  A slot is corrected by
one link, the last listed, from the uncorrected populations
(bouzidi_kernel.jl:13-92 writes each slot anew from f_post_collision), so the
first listings change nothing: not the number of links (their share of the
footprint, no device needed), and not the fields.

Device: 1,500 cells with every direction cut, listed twice, with the same
distances and with other ones in the first listing, against the oracle's loop
over the same list; strict build, bit-identical."""
import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from openludwig_amd.solver import footprint
from parity_helpers import compare, run_pair
from test_gpu_boundary_blocks import _box
from test_gpu_wall_links import _cut


def _listed_twice(level, other):
    q = level.bouzidi_q
    first = np.random.default_rng(5).permutation(q, axis=0) if other else q
    # every link of the second listing exists in the first one too, and the other way round
    first = np.where((q.view(np.float16) > 0) & (first.view(np.float16) > 0), first, q).astype(np.uint16)
    level.bouzidi_cells = np.concatenate([level.bouzidi_cells, level.bouzidi_cells])
    level.bouzidi_q = np.ascontiguousarray(np.concatenate([first, q]))
    level.bouzidi_tri = np.zeros(level.bouzidi_q.shape, np.int32)


def _config():
    cfg, _ = cases.tiny_sphere(8, 1, ddf=True)
    return cfg.replace(ramp_steps=2, forces_enabled=False, limiter="none")


@pytest.mark.parametrize("other", [False, True])
def test_listings_do_not_add_links(other):
    cfg = _config()
    grids, params = _box(3, 1, 1)
    _cut(grids[0], 1, 11)
    once = footprint(cfg, grids, params, None)
    _listed_twice(grids[0], other)
    assert footprint(cfg, grids, params, None) == once


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16])
@pytest.mark.parametrize("other", [False, True])
def test_last_listing_counts_strict_bitexact(hip_device, other, storage):
    cfg = _config()
    grids, params = _box(3, 1, 1)
    _cut(grids[0], 1, 11)
    _listed_twice(grids[0], other)
    s, o = run_pair(cfg, grids, params, None, steps=2, strict=True, batch=2, storage=storage, amp=0.02)
    res = compare(s, o, grids, ("f", "rho", "vel", "g", "T"))
    s.close()
    o.close()
    for k, (mx, n, _) in res.items():
        assert mx == 0.0, f"other distances {other} {k}: max |diff| {mx} over {n} entries"
