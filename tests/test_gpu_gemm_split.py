"""GPU parity of the prefill GEMMs with K split over workgroups (calls of few
tiles): ranges of unequal length, K not a multiple of 256 or 64, odd N, weights
off 16 bytes, the gate/up pair, subnormal block scales at range ends, rows of
extreme size and non-finite rows. Bound as for the unsplit GEMM: 2e-3 *
||x_b|| * ||w_r|| per element.
"""
import numpy as np
import pytest

import kunlunk200_lib_amd as kl
from gpu_util import run_matmul, weight_payload
from test_gpu_decode_edges import gemm_bound_ok, q4_sparse_subnormal, q4_subnormal
from test_gpu_gemm import check_gemm, gaussian
from test_gpu_swiglu import check_pair, run_pair

pytestmark = pytest.mark.gpu

Q4, F16 = kl.WeightType.q4_0, kl.WeightType.f16

# (type, k, n, batch, w_offset): the LDS-copy kernel takes Q4_0 with K % 256 == 0 and
# 16-byte aligned weights, the register-staged one the rest
SHAPES = [(Q4, 4096, 300, 64, 0), (Q4, 2304, 1, 65, 0), (Q4, 16384, 129, 130, 0), (Q4, 2048, 1000, 100, 0),
          (Q4, 5600, 131, 77, 0), (Q4, 1312, 64, 200, 0), (Q4, 4096, 257, 70, 2), (Q4, 16352, 33, 64, 1),
          (F16, 4096, 300, 64, 0), (F16, 5600, 2999, 77, 0), (F16, 1312, 1, 129, 0), (F16, 16384, 65, 256, 0)]


@pytest.mark.parametrize("wtype,k,n,batch,w_offset", SHAPES)
def test_split_gemm(gpu, oracle, wtype, k, n, batch, w_offset):
    w = gaussian((n, k), 0.02, k + n)
    x = gaussian((batch, k), 1.0, k + n + 1)
    x[3] *= 1e6
    x[7] *= 1e-30
    x[9, : k // 2] *= 1e4
    payload, dec = weight_payload(wtype, w, oracle)
    y, route, guard_ok = run_matmul(wtype, payload, x, k, n, batch, w_offset=w_offset)
    finite, ok, _ = check_gemm(y, oracle.gold(dec, x, threads=16), dec, x)
    assert route == ("q4_gemm_mfma" if wtype == Q4 else "f16_gemm_mfma") and guard_ok and finite and ok


@pytest.mark.parametrize("k,n,batch", [(4096, 300, 64), (5600, 131, 77)])
def test_split_gemm_nonfinite_rows(gpu, oracle, k, n, batch):
    # a non-finite activation in one K range makes its row non-finite and no other
    x = gaussian((batch, k), 1.0, 5)
    x[1, 3], x[2, k - 1] = np.nan, -np.inf
    payload, dec = weight_payload(Q4, gaussian((n, k), 0.02, 6), oracle)
    y, _, guard_ok = run_matmul(Q4, payload, x, k, n, batch)
    assert guard_ok and not np.any(np.isfinite(y[1:3])) and np.all(np.isfinite(np.delete(y, (1, 2), axis=0)))


@pytest.mark.parametrize("wtype,k,n,batch", [(Q4, 4096, 300, 64), (Q4, 2304, 67, 130), (Q4, 5600, 131, 77), (F16, 4096, 129, 70)])
def test_split_gemm_pair(gpu, oracle, wtype, k, n, batch):
    x = gaussian((batch, k), 1.0, 3)
    pg, dg = weight_payload(wtype, gaussian((n, k), 0.02, 1), oracle)
    pu, du = weight_payload(wtype, gaussian((n, k), 0.02, 2), oracle)
    y, route = run_pair(wtype, pg, pu, x, k, n, batch)
    finite, ok, worst = check_pair(y, x, dg, du, oracle, 2e-3)
    assert route == ("q4" if wtype == Q4 else "f16") + "_gemm_swiglu_mfma" and finite and ok, worst


@pytest.mark.parametrize("k,n,batch,sparse", [(4096, 700, 100, True), (4096, 200, 100, False), (5600, 150, 77, True),
                                              (5600, 150, 77, False)])
def test_split_gemm_subnormal_scales(gpu, oracle, k, n, batch, sparse):
    q4 = q4_sparse_subnormal(k, n, 97) if sparse else q4_subnormal(k, n, 91, True, tiny=True)
    dec = oracle.q4_decode(q4, k, n)
    x = np.random.default_rng(98).standard_normal((batch, k)).astype(np.float32)
    y, _, guard_ok = run_matmul(Q4, q4, x, k, n, batch)
    assert guard_ok and np.all(np.isfinite(y))
    ok, ratio = gemm_bound_ok(y, oracle.gold(dec, x, threads=16), dec, x, 2e-3)
    assert ok, f"error {ratio:.3g} x the bound"


@pytest.mark.parametrize("k,n,batch", [(4096, 150, 70), (5600, 150, 77)])
def test_split_gemm_pair_subnormal_scales(gpu, oracle, k, n, batch):
    pg, pu = q4_sparse_subnormal(k, n, 11), q4_sparse_subnormal(k, n, 12)
    x = np.random.default_rng(13).standard_normal((batch, k)).astype(np.float32)
    y, route = run_pair(Q4, pg, pu, x, k, n, batch)
    finite, ok, worst = check_pair(y, x, oracle.q4_decode(pg, k, n), oracle.q4_decode(pu, k, n), oracle, 2e-3)
    assert route == "q4_gemm_swiglu_mfma" and finite and ok, worst
