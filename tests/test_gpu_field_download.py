"""Field downloads through the pinned ring: one row, rows that end inside a
piece, more pieces than the ring holds, and contexts that download at the same
time from several threads; the caller's block order, all fields and storages.

An uploaded field comes back as it is stored: FP32 to the bit, 16-bit
populations as w_k + round(f - w_k) (numpy's binary16 rounding, torch's bfloat16
cast, both pinned against the oracle elsewhere)."""
import threading

import numpy as np
import pytest
import torch

from openludwig_amd import _native as N
from openludwig_amd import cases
from openludwig_amd.solver import Solver
from parity_helpers import _weights
from test_gpu_boundary_blocks import _box


def _stored(f, storage):
    w = _weights()[:, None]
    d = (f - w).astype(np.float32)
    if storage == N.LB_STORAGE_FP16:
        return w + d.astype(np.float16).astype(np.float32)
    if storage == N.LB_STORAGE_BF16:
        return w + torch.from_numpy(d).to(torch.bfloat16).to(torch.float32).numpy()
    return f


def _case(shape, storage, seed):
    cfg, _ = cases.tiny_sphere(8, 1, ddf=True)
    grids, params = _box(*shape)
    s = Solver(cfg.replace(forces_enabled=False), grids, params, None, storage=storage)
    s.init_equilibrium()
    rng = np.random.default_rng(seed)
    n = grids[0].n_cells
    want = {}
    for name, comps in (("f", 27), ("g", 27), ("rho", 1), ("vel", 3), ("T", 1)):
        a = rng.standard_normal((comps, n)).astype(np.float32)
        if comps == 27:
            a = (_weights()[:, None] * (1 + 0.1 * a)).astype(np.float32)
        s.upload(1, name, a.ravel())
        want[name] = (_stored(a, storage) if comps == 27 else a).ravel()
    return s, want


@pytest.mark.gpu
@pytest.mark.parametrize("storage", [N.LB_STORAGE_FP32, N.LB_STORAGE_FP16, N.LB_STORAGE_BF16])
@pytest.mark.parametrize("shape", [(1, 1, 1), (5, 3, 2), (13, 11, 7)])
def test_download_returns_what_is_stored(hip_device, shape, storage):
    s, want = _case(shape, storage, 5)
    for name, a in want.items():
        assert np.array_equal(s.download(1, name), a), name
    s.close()


@pytest.mark.gpu
def test_downloads_from_several_threads(hip_device):
    made = [_case((7, 5, 4), storage, 20 + i) for i, storage in enumerate((0, 1, 2, 0))]
    wrong = []

    def read(s, want):
        for _ in range(3):
            for name, a in want.items():
                if not np.array_equal(s.download(1, name), a):
                    wrong.append(name)

    threads = [threading.Thread(target=read, args=m) for m in made]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s, _ in made:
        s.close()
    assert not wrong
