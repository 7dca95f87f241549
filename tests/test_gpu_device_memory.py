"""What a case holds against what it counts: the device memory that creating a
case takes from the pool is no more than lb_device_bytes, and nothing is
allocated only to reach that count (the link records take 16 bytes of the 24
that a link counts)."""
import ctypes as C

import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from openludwig_amd.solver import Solver, build_case

USED_MEM_CURRENT = 7  # hipMemPoolAttrUsedMemCurrent


def _used() -> int:
    hip = N.hip_lib()  # the runtime that the library is bound to
    pool, used = C.c_void_p(), C.c_uint64()
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    assert hip.hipMemPoolGetAttribute(pool, USED_MEM_CURRENT, C.byref(used)) == 0
    return used.value


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16])
def test_a_case_allocates_no_padding(hip_device, storage):
    cfg, mesh = cases.sphere_re1e3(16, 3)
    grids, params, mesh = build_case(cfg, mesh)
    q = [g.bouzidi_q.view(np.float16).astype(np.float32) for g in grids]
    links = sum(int(np.count_nonzero((a > cfg.q_min_threshold) & (a <= 1.0))) for a in q)
    assert links > 10_000
    before = _used()
    s = Solver(cfg, grids, params, mesh, storage=storage)
    held, counted = _used() - before, s.device_bytes
    s.close()
    assert _used() == before
    assert held > 0.9 * counted
    # the pool rounds each of the case's about 100 buffers up, by less than 64 bytes
    assert held <= counted - 8 * links + 64 * 150, (held, counted, links)
