"""One-sided direct forces where the source chunks' rule drops the last chunk or keeps
it (gravity.hip, pick_chunks), on device arrays, through the caller's workspace with
a guard behind it.  Against sums in extended precision on sampled rows, 1e-14 of
sum_j |a_ij| (split 4e-7), as in test_gpu_direct_split.py."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_active", [(27548, 27548), (30011, 20011), (34972, 17486), (18332, 9166), (16628, 16245),
                                        (25105, 6705), (58268, 29134), (8348, 8348)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-14), ("split", 4e-7)])
def test_chunk_rule(gpu, n, n_active, precision, tol):
    hip = ctypes.CDLL("libamdhip64.so", mode=ctypes.RTLD_GLOBAL)
    L = gpu.lib()
    rng = np.random.default_rng(n)
    h = np.concatenate([rng.normal(size=(3, n)), rng.uniform(0.1, 2.0, (1, n)) / n])
    ws_bytes = L.reb_amd_gravity_workspace_bytes(n, gpu.PRECISION[precision])
    dev, ws = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(dev), ctypes.c_size_t(7 * 8 * n)) == 0
    assert hip.hipMalloc(ctypes.byref(ws), ctypes.c_size_t(ws_bytes + 4096)) == 0
    guard = np.full(512, 7.25)
    assert hip.hipMemcpy(dev, h.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(h.nbytes), 1) == 0
    assert hip.hipMemcpy(ctypes.c_void_p(ws.value + ws_bytes), guard.ctypes.data_as(ctypes.c_void_p),
                         ctypes.c_size_t(4096), 1) == 0
    p = [dev.value + 8 * n * k for k in range(7)]
    assert L.reb_amd_gravity_direct(*p, n, n_active, 0, 0, 1.0, 0.01, gpu.PRECISION[precision], 0, ws.value, None) == 0
    acc, after = np.zeros((3, n)), np.zeros(512)
    assert hip.hipMemcpy(acc.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(p[4]), ctypes.c_size_t(acc.nbytes), 2) == 0
    assert hip.hipMemcpy(after.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(ws.value + ws_bytes),
                         ctypes.c_size_t(4096), 2) == 0
    assert hip.hipFree(dev) == 0 and hip.hipFree(ws) == 0
    assert np.array_equal(after, guard)
    x, m = h[:3, :n_active].astype(np.longdouble), h[3, :n_active]
    for i in (0, 1, 255, 256, n_active - 1, n // 2, n - 257, n - 1):
        d = x - h[:3, i:i + 1]
        r2 = (d * d).sum(0) + np.longdouble(0.01) ** 2
        terms = m * d / (r2 * np.sqrt(r2))
        assert np.sqrt(((acc[:, i] - terms.sum(1)) ** 2).sum()) <= tol * np.sqrt((terms * terms).sum(0)).sum()
