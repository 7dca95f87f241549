"""A context with queued steps holds up nobody else: a field download of that
context, which waits for its steps, leaves other contexts' downloads, creation
and destruction free (they share pinned memory and the device's hardware
queues).  Fields downloaded beside queued steps come another way than alone
(copies, reordered and decoded by the host's threads) and are the same: FP32 to
the bit, 16-bit populations as w_k + round(f - w_k), from one block to more
pieces than there are."""
import threading
import time

import numpy as np
import pytest

from openludwig_amd import _native as N
from openludwig_amd import cases
from openludwig_amd.solver import Solver, build_case
from test_gpu_field_download import _case

STEPS = 2500  # about 0.4 s more than it takes to queue them


@pytest.fixture(scope="module")
def sphere():
    cfg, mesh = cases.sphere_re1e3(16, 3)
    return cfg, *build_case(cfg, mesh)


def _queue_steps(sphere):
    s = Solver(*sphere)
    s.init_equilibrium()
    s.download(1, "rho")
    s.execute_timestep_batch(1, 1, 0.05)
    s.synchronize()
    s.execute_timestep_batch(2, STEPS, 0.05)
    return s


@pytest.mark.gpu
def test_others_go_on_beside_a_busy_context(hip_device, sphere):
    # more contexts than hardware queues: some streams share the busy one's
    others = [Solver(*sphere) for _ in range(6)]
    for s in others:
        s.init_equilibrium()
        s.download(1, "rho")
    busy = _queue_steps(sphere)
    last = threading.Thread(target=lambda: busy.download(1, "rho"))
    last.start()
    waiting = []
    for s in others:
        rho, vel = s.download(1, "rho"), s.download(3, "vel")
        assert np.all(rho == 1.0) and np.all(vel == 0.0)
        waiting.append(last.is_alive())
    Solver(*sphere).close()
    waiting.append(last.is_alive())
    last.join()
    for s in (*others, busy):
        s.close()
    assert all(waiting), waiting


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16, N.LB_STORAGE_BF16])
@pytest.mark.parametrize("shape", [(1, 1, 1), (5, 3, 2), (13, 11, 7)])
def test_fields_beside_a_busy_context(hip_device, sphere, shape, storage):
    s, want = _case(shape, storage, 5)
    busy = _queue_steps(sphere)
    got = {name: s.download(1, name) for name in want}
    t = time.perf_counter()
    busy.synchronize()
    waited = time.perf_counter() - t
    busy.close()
    s.close()
    assert waited > 1e-3, "the steps were done before the downloads"
    for name, a in want.items():
        assert np.array_equal(got[name], a), name
