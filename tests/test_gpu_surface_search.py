"""The shell search of the surface probe (map_stresses_kernel!,
surface.jl:395-452) for triangles whose probes meet no fluid: search radii from
one shell to rows of 17 cells (four blocks), a body that leaves the level's
blocks and the domain on its low and high side, and both sides of the surface
(inside the solid body no shell may hold a fluid cell).

Strict build against the oracle's loop over the shells: per-triangle pressure
and shear bit-identical."""
import ctypes as C

import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from openludwig_amd.solver import build_case
from parity_helpers import run_pair


def _oracle_maps(o, cfg, params, mesh, dx, radius, offset, side):
    f32 = np.float32
    arr = [np.ascontiguousarray(a, dtype=f32) for a in
           (mesh.centers[:, 0], mesh.centers[:, 1], mesh.centers[:, 2], side * mesh.normals[:, 0],
            side * mesh.normals[:, 1], side * mesh.normals[:, 2], mesh.areas)]
    off, ref = np.array(offset, f32), np.array(params.moment_center, f32)
    ps = float(f32(params.rho_physical * params.velocity_scale * params.velocity_scale))
    out, maps = np.zeros(9), np.zeros(4 * mesh.n, f32)
    p = lambda a, t: a.ctypes.data_as(C.POINTER(t))  # noqa: E731
    o.L.orc_forces(o.ctx, 0, *[p(a, C.c_float) for a in arr], mesh.n, p(off, C.c_float), p(ref, C.c_float),
                   float(f32(dx)), ps, ps, radius, cfg.c_wale, cfg.nu_sgs_background, p(out, C.c_double),
                   p(maps, C.c_float))
    return maps.reshape(4, mesh.n)


@pytest.mark.gpu
def test_search_strict_bitexact(hip_device):
    cfg, mesh = cases.tiny_sphere(8, 2)
    grids, params, mesh = build_case(cfg, mesh)
    s, o = run_pair(cfg, grids, params, mesh, steps=6, strict=True)
    size = params.domain_size
    for shift in ((0.0, 0.0, 0.0), (-1.9, 0.1, -1.4), (size[0] - 2.2, 0.03, size[2] - 2.6)):
        offset = tuple(params.mesh_offset[i] + shift[i] for i in range(3))
        for radius in (1, 3, 5, 8):
            for side in (1, -1):
                fp = s._force_params()
                fp.search_radius = radius
                for i in range(3):
                    fp.mesh_offset[i] = offset[i]
                got = [np.zeros(mesh.n, np.float32) for _ in range(4)]
                assert s.lib.lb_surface_maps(s._ctx, C.byref(fp), side, *[N.ptr(m, C.c_float) for m in got]) == 0
                want = _oracle_maps(o, cfg, params, mesh, grids[-1].dx, radius, offset, side)
                for i in range(4):
                    assert np.array_equal(got[i], want[i]), f"shift {shift} radius {radius} side {side} map {i}"
    s.close()
    o.close()
