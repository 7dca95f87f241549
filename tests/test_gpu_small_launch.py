"""Occupancy of 16-bit stream-collide launches: up to 1,280 blocks run the build
for 5 waves per SIMD, larger ones the build for 6.  Boxes of one level on both
sides of the line.

Strict build against the FP32 oracle from the same perturbed state: both builds
round every operation alike, so all fields are bit-identical."""
import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from parity_helpers import compare, run_pair
from test_gpu_boundary_blocks import _box


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP16, N.LB_STORAGE_BF16])
@pytest.mark.parametrize("shape", [(16, 10, 8), (61, 3, 7)])  # 1,280 and 1,281 blocks
def test_line_strict_bitexact(hip_device, shape, storage):
    cfg, _ = cases.tiny_sphere(8, 1)
    cfg = cfg.replace(inlet_turbulence_intensity=np.float32(0.01), ramp_steps=2, boundary_method="none",
                      forces_enabled=False)
    grids, params = _box(*shape)
    s, o = run_pair(cfg, grids, params, None, steps=2, strict=True, batch=2, storage=storage, amp=0.02)
    res = compare(s, o, grids, ("f", "rho", "vel"))
    s.close()
    o.close()
    for k, (mx, n, _) in res.items():
        assert mx == 0.0, f"{shape} {k}: max |diff| {mx} over {n} entries"
