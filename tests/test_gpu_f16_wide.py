"""GPU parity of the wide F16 prefill tiles (256 and 128 activation rows x 256
weight rows, forced by KUNLUN_GEMM_TILE=256x64 and 128x64): one to many K steps
(odd and even counts, K % 64 == 32 on the 256-row tile), partial row and column
tiles, the gate/up pair, extreme F16 values and rows, non-finite weights.
Bound as for the other GEMM tiles: 2e-3 * ||x_b|| * ||w_r|| per element.
"""
import numpy as np
import pytest

import kunlunk200_lib_amd as kl
from gpu_util import run_matmul, weight_payload
from test_gpu_gemm import check_gemm, gaussian
from test_gpu_swiglu import check_pair, run_pair

pytestmark = pytest.mark.gpu

F16 = kl.WeightType.f16
WIDE = ["256x64", "128x64"]


@pytest.mark.parametrize("tile", WIDE)
@pytest.mark.parametrize("k,n,batch", [(32, 64, 64), (64, 700, 200), (96, 33, 70), (192, 257, 129), (4096, 300, 513),
                                       (320, 1, 256), (16384, 256, 65), (5600, 511, 300)])
def test_f16_wide_tiles(gpu, oracle, knobs, tile, k, n, batch):
    knobs("KUNLUN_GEMM_TILE", tile)
    w = gaussian((n, k), 0.02, k + n)
    w[0] *= 1e5                                # up to the largest F16 values
    w[n // 2] *= 1e-4                          # and into its subnormals
    x = gaussian((batch, k), 1.0, k + n + 1)
    x[3] *= 1e6
    x[7] *= 1e-30
    payload, dec = weight_payload(F16, w, oracle)
    y, route, guard_ok = run_matmul(F16, payload, x, k, n, batch)
    finite, ok, _ = check_gemm(y, oracle.gold(dec, x, threads=16), dec, x)
    assert route == "f16_gemm_mfma" and guard_ok and finite and ok


@pytest.mark.parametrize("tile", WIDE)
@pytest.mark.parametrize("k,n,batch", [(512, 300, 130), (4096, 129, 300), (96, 127, 257)])
def test_f16_wide_pair(gpu, oracle, knobs, tile, k, n, batch):
    knobs("KUNLUN_GEMM_TILE", tile)
    x = gaussian((batch, k), 1.0, 3)
    pg, dg = weight_payload(F16, gaussian((n, k), 0.02, 1), oracle)
    pu, du = weight_payload(F16, gaussian((n, k), 0.02, 2), oracle)
    y, route = run_pair(F16, pg, pu, x, k, n, batch)
    finite, ok, worst = check_pair(y, x, dg, du, oracle, 2e-3)
    assert route == "f16_gemm_swiglu_mfma" and finite and ok, worst


@pytest.mark.parametrize("tile", WIDE)
def test_f16_wide_nonfinite(gpu, oracle, knobs, tile):
    # a non-finite weight touches its output column alone, a non-finite activation its row
    knobs("KUNLUN_GEMM_TILE", tile)
    k, n, batch = 320, 300, 200
    w = gaussian((n, k), 0.02, 5)
    w[n - 1, k - 1], w[40, 0] = np.inf, np.nan
    x = gaussian((batch, k), 1.0, 6)
    x[batch - 1, k - 1] = np.nan
    payload, _ = weight_payload(F16, w, oracle)
    y, _, guard_ok = run_matmul(F16, payload, x, k, n, batch)
    bad = np.zeros((batch, n), bool)
    bad[batch - 1], bad[:, n - 1], bad[:, 40] = True, True, True
    assert guard_ok and np.array_equal(~np.isfinite(y), bad)
