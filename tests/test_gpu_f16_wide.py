"""GPU parity of the wide F16 prefill tiles (256 and 128 activation rows x 256
weight rows, forced by KUNLUN_GEMM_TILE=256x64 and 128x64, and by the dispatch;
sums that show which kernel ran): one to many K steps
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


# Sums that tell the kernels apart (all take the same route): 2^30 at K 0 and -2^30 in the
# fourth last K32 block, ones in `blocks`. An F32 chain that holds 2^30 drops the ones added to
# it (half a unit there is 64, an MFMA adds at most 32), one without it keeps them.
def order_probe(k, n, batch, blocks):
    x, w = np.zeros((batch, k // 32, 32), np.float32), np.ones((n, k), np.float32)
    x[:, blocks] = 1.0
    x = x.reshape(batch, k)
    at = k - 128
    x[:, 0] = x[:, at] = 2.0**15
    w[:, 0], w[:, at] = 2.0**15, -(2.0**15)
    y, route, guard_ok = run_matmul(F16, w.astype(np.float16).view(np.uint8), x, k, n, batch)
    assert route == "f16_gemm_mfma" and guard_ok
    return y


def rows_256(k, n, batch):
    # one chain over all of K: 31 ones at most beside -2^30, and the last three blocks
    y = order_probe(k, n, batch, slice(None))
    return bool(np.all((y >= 96) & (y <= 128)))


def rows_128(k, n, batch):
    # a chain of the even blocks (with 2^30) and one of the odd ones; the register-staged
    # kernel has blocks 0, 1 of every four in one chain, a split has whole ranges
    return bool(np.all(order_probe(k, n, batch, slice(1, None, 4)) == k // 128 * 32))


@pytest.mark.parametrize("k,n,batch", [(4096, 300, 513), (5632, 511, 300), (16384, 256, 65), (4096, 11008, 512)])
def test_f16_forced_tile_runs(gpu, knobs, k, n, batch):
    knobs("KUNLUN_GEMM_TILE", "256x64")
    assert rows_256(k, n, batch) and not rows_128(k, n, batch)
    knobs("KUNLUN_GEMM_TILE", "128x64")
    assert rows_128(k, n, batch) and not rows_256(k, n, batch)
    knobs("KUNLUN_GEMM_TILE", "128x48")            # another tile: no wide one
    assert not rows_128(k, n, batch) and not rows_256(k, n, batch)


# Calls that the dispatch gives to the wide tiles (128 and 256 rows) by itself
@pytest.mark.parametrize("k,n,batch,runs", [(4096, 11008, 512, rows_128), (4096, 11008, 1024, rows_256)])
def test_f16_wide_dispatch(gpu, oracle, k, n, batch, runs):
    assert runs(k, n, batch)
    x = gaussian((batch, k), 1.0, 8)
    payload, dec = weight_payload(F16, gaussian((n, k), 0.02, 9), oracle)
    y, route, guard_ok = run_matmul(F16, payload, x, k, n, batch)
    some = np.r_[0:40, 4000:4100, n - 40:n]
    finite, ok, _ = check_gemm(y[:, some], oracle.gold(dec[some], x, threads=16), dec[some], x)
    assert route == "f16_gemm_mfma" and guard_ok and finite and ok and np.all(np.isfinite(y))


# One round of register-staged tiles stays there from K 192 on, two rounds do not (the probe needs K 256)
@pytest.mark.parametrize("k,n,batch,runs", [(256, 1000, 512, False), (384, 16384, 100, False), (256, 9434, 222, True)])
def test_f16_short_k_dispatch(gpu, k, n, batch, runs):
    assert rows_128(k, n, batch) == runs


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
