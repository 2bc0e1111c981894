"""GPU parity of the F32 GEMM (F32 weights, more than 16 columns, route
f32_mfma_gemv): partial row, column and K tiles, one and two workgroups per CU,
and special values, which follow F32 arithmetic.

Bound: the F32-accumulate GEMV's, |y - gold| <= 1e-4 * ||x_b|| * ||w_r||, gold
the FP64 dot; the error against gold stays below 1e-6 of its norm.
"""
import numpy as np
import pytest

import kunlunk200_lib_amd as kl
from gpu_util import check_f32_accumulate, run_matmul

pytestmark = pytest.mark.gpu

F32 = kl.WeightType.f32


@pytest.mark.parametrize("k,n,batch", [(32, 7, 17), (96, 40, 33), (1056, 65, 70), (160, 5000, 30), (4096, 300, 100),
                                       (16384, 17, 64), (256, 4200, 65), (1152, 16, 32), (1056, 40, 33),
                                       (8192, 65, 33), (4096, 1024, 33), (4096, 1, 17), (1152, 15, 48), (96, 3, 49)])
def test_f32_gemm_shapes(gpu, oracle, k, n, batch):
    rng = np.random.default_rng(k + n + batch)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    x = rng.standard_normal((batch, k)).astype(np.float32)
    y, route, guard_ok = run_matmul(F32, w.view(np.uint8), x, k, n, batch)
    gold = oracle.gold(w, x, threads=16)
    res = check_f32_accumulate(y, gold, w, x)
    print(f"  f32 gemm k={k} n={n} b={batch} {res}", flush=True)
    assert route == "f32_mfma_gemv" and guard_ok and res["finite"] and res["north_star"] and res["reference"]
    assert np.linalg.norm(y - gold) <= 1e-6 * np.linalg.norm(gold)


def test_f32_gemm_special_values(gpu):
    k, n, batch = 288, 40, 70
    rng = np.random.default_rng(4)
    w = rng.standard_normal((n, k)).astype(np.float32)
    x = (np.abs(rng.standard_normal((batch, k))) + 0.5).astype(np.float32)
    w[3, 270], w[4, 5], w[5, 100] = np.inf, -np.inf, np.nan
    x[66, 280] = np.nan
    y, _, guard_ok = run_matmul(F32, w.view(np.uint8), x, k, n, batch)
    rest = np.delete(y, 66, axis=0)
    assert guard_ok and np.all(np.isnan(y[66]))
    assert np.all(rest[:, 3] == np.inf) and np.all(rest[:, 4] == -np.inf) and np.all(np.isnan(rest[:, 5]))
    assert np.all(np.isfinite(np.delete(rest, (3, 4, 5), axis=1)))
