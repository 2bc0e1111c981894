"""GPU parity of the K-split Q4_0 MFMA GEMV (3..32 columns per pass, route
q4_mfma_gemv) and its gate/up pair: partial last steps and blocks (K % 256,
K % 64), weights and activations off their natural alignment, one and several
K ranges and LDS chunks, tiles of several rounds, and the cap on partial sums.

Bound: the F32-accumulate GEMV's, |y - gold| <= 1e-4 * ||x_b|| * ||w_r||, gold
the FP64 dot of the exactly decoded weights.
"""
import numpy as np
import pytest

import kunlunk200_lib_amd as kl
from gpu_util import check_f32_accumulate, run_matmul
from test_gpu_swiglu import check_pair, device_swiglu, run_pair

pytestmark = pytest.mark.gpu

Q4 = kl.WeightType.q4_0

SPLIT, GENERAL = "q4_mfma_gemv", "gemv_general"

# (k, n, batch, w_offset, x_offset, route): the route of the first pass of 32 columns
SHAPES = [(32, 7, 9, 0, 0, SPLIT), (96, 33, 17, 0, 0, SPLIT), (1056, 65, 24, 0, 0, SPLIT),      # K % 64 == 32
          (544, 7000, 3, 0, 0, SPLIT), (4128, 70, 4, 0, 0, SPLIT),
          # misaligned
          (2048, 129, 20, 2, 0, SPLIT), (1024, 50, 12, 1, 0, SPLIT), (5120, 40, 7, 3, 4, SPLIT), (4096, 33, 31, 4, 8, SPLIT),
          (4096, 16, 16, 0, 0, SPLIT), (4096, 17, 32, 0, 0, SPLIT), (4096, 300, 33, 0, 0, SPLIT), (4096, 300, 63, 0, 0, SPLIT),
          (11008, 257, 8, 0, 0, SPLIT), (11008, 40, 12, 0, 0, SPLIT), (16384, 48, 32, 0, 0, SPLIT),
          (2304, 33000, 32, 0, 0, SPLIT), (512, 20000, 30, 0, 0, SPLIT), (8192, 1, 5, 0, 0, SPLIT),
          # more row tiles per workgroup than it has waves: a second round on the same fragments
          (4096, 17000, 32, 0, 0, SPLIT), (544, 66000, 9, 0, 0, SPLIT), (1056, 65600, 8, 0, 0, SPLIT),
          # shapes off the batch-1 kernels with little work: a wave's row per pass of 64 blocks and 8 columns
          (544, 70, 3, 0, 0, GENERAL), (512, 40, 7, 3, 4, GENERAL), (1056, 1000, 8, 0, 0, GENERAL), (1056, 1000, 9, 0, 0, SPLIT),
          (2976, 300, 5, 0, 0, GENERAL), (2976, 300, 6, 0, 0, SPLIT), (2976, 1100, 3, 0, 0, SPLIT)]


@pytest.mark.parametrize("k,n,batch,w_offset,x_offset,expected", SHAPES)
def test_split_shapes(gpu, oracle, k, n, batch, w_offset, x_offset, expected):
    rng = np.random.default_rng(k + 3 * n + batch)
    q4 = kl.quantize_q4_0((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((batch, k)).astype(np.float32)
    x[batch - 1] *= 1e-20                      # each column and step has its own scale
    x[0, : k // 2] *= 1e8
    y, route, guard_ok = run_matmul(Q4, q4, x, k, n, batch, w_offset=w_offset, x_offset=x_offset)
    dec = oracle.q4_decode(q4, k, n)
    res = check_f32_accumulate(y, oracle.gold(dec, x, threads=16), dec, x)
    print(f"  split k={k} n={n} b={batch} route={route} {res}", flush=True)
    assert route == expected
    assert guard_ok and res["finite"] and res["north_star"]


# the knobs' batch range holds above 16 columns too
@pytest.mark.parametrize("knob,value", [("KUNLUN_Q4_MFMA_MIN", "17"), ("KUNLUN_Q4_MFMA_MAX", "15")])
@pytest.mark.parametrize("k,route", [(4096, "q4_gemv_dot8"), (1056, GENERAL)])
def test_split_off_by_knob(gpu, oracle, knobs, knob, value, k, route):
    n, batch = 70, 32
    rng = np.random.default_rng(k)
    q4 = kl.quantize_q4_0((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((batch, k)).astype(np.float32)
    knobs(knob, value)
    y, taken, guard_ok = run_matmul(Q4, q4, x, k, n, batch)
    dec = oracle.q4_decode(q4, k, n)
    res = check_f32_accumulate(y, oracle.gold(dec, x, threads=16), dec, x)
    assert taken == route and guard_ok and res["finite"] and res["north_star"]


# (k, batch, w_offset): 3..63 columns with K % 64 != 0 or weights off a dword follow F32
# arithmetic in an infinite activation, the others make its column NaN
@pytest.mark.parametrize("k,batch,w_offset", [(4096, 20, 0), (11008, 6, 0), (4160, 7, 0), (1056, 12, 0), (5600, 5, 0),
                                              (1056, 40, 0), (512, 9, 2), (4096, 17, 1), (4128, 4, 0), (96, 3, 0)])
def test_split_nonfinite(gpu, oracle, k, batch, w_offset):
    # a non-finite activation touches its column and no other; an infinite block
    # scale makes its row's outputs infinite or NaN and no other's
    n = 40
    rng = np.random.default_rng(k)
    q4 = kl.quantize_q4_0((rng.standard_normal((n, k)) * 0.02).astype(np.float32)).reshape(n, k // 32, 18)
    q4[5, k // 32 - 1, :2] = np.array([np.inf], np.float16).view(np.uint8)
    q4[6, k // 32 - 1, :2] = 0
    q4[7, k // 32 - 1, 17] = 0x88                  # weight 0 at K - 1
    x = rng.standard_normal((batch, k)).astype(np.float32)
    x[0] *= 1e30
    x[1, 3], x[2, k - 1] = np.nan, -np.inf
    x[batch - 1, :2] = np.inf, np.inf
    x[batch - 1, 40] = 1e37
    payload = q4.reshape(n, -1)
    y, _, guard_ok = run_matmul(Q4, payload, x, k, n, batch, w_offset=w_offset)
    rows = np.arange(n) != 5
    assert guard_ok and np.all(np.isnan(y[1]))
    rest = np.delete(y, (1, 2, batch - 1), axis=0)
    assert np.all(np.isfinite(rest[:, rows])) and not np.any(np.isfinite(rest[:, 5]))
    w = oracle.q4_decode(payload, k, n).astype(np.float64)
    if k % 64 == 0 and w_offset % 4 == 0:
        assert np.all(np.isnan(y[2])) and np.all(np.isnan(y[batch - 1]))
        return
    for col in {2, batch - 1}:
        with np.errstate(invalid="ignore"):
            want = (w[rows] * x[col].astype(np.float64)).sum(1)
        got = y[col][rows]
        assert not np.any(np.isfinite(want)) and np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(got[~np.isnan(want)], want[~np.isnan(want)].astype(np.float32)) and np.any(np.isinf(want))


@pytest.mark.parametrize("k,batch", [(4096, 20), (11008, 6), (1056, 12)])
def test_split_largest_activations(gpu, oracle, k, batch):
    # up to the largest F32 value, whose product with a small weight is finite
    n = 40
    rng = np.random.default_rng(k + 1)
    q4 = kl.quantize_q4_0((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((batch, k)).astype(np.float32)
    x[1, 3], x[2, k - 1], x[batch - 1, 300] = np.finfo(np.float32).max, -np.finfo(np.float32).max, 2.0**127
    y, _, guard_ok = run_matmul(Q4, q4, x, k, n, batch)
    dec = oracle.q4_decode(q4, k, n)
    res = check_f32_accumulate(y, oracle.gold(dec, x, threads=16), dec, x)
    assert guard_ok and res["finite"] and res["north_star"]


# the second line: second rounds, with one k-group and with four (which use their exchange
# area again), in one K range and in several; the third: one range, whose products and
# SwiGLU are one launch, with one to eight k-groups and one to three rounds
@pytest.mark.parametrize("k,n,batch", [(1056, 65, 24), (4096, 300, 32), (11008, 50, 5), (2048, 1000, 30), (96, 20, 40),
                                       (4096, 4096, 16), (4096, 4090, 32), (2080, 4200, 8), (1056, 8500, 12), (4096, 8300, 32),
                                       (1536, 1000, 16), (1536, 4097, 9), (544, 300, 12), (32, 50, 16), (2080, 17, 10),
                                       (512, 66000, 17), (1024, 9000, 32), (1056, 33000, 8)])
def test_split_pair(gpu, oracle, k, n, batch):
    rng = np.random.default_rng(k + n + batch)
    pg, pu = (kl.quantize_q4_0((rng.standard_normal((n, k)) * 0.02).astype(np.float32)) for _ in range(2))
    x = rng.standard_normal((batch, k)).astype(np.float32)
    y, route = run_pair(Q4, pg, pu, x, k, n, batch)
    finite, ok, worst = check_pair(y, x, oracle.q4_decode(pg, k, n), oracle.q4_decode(pu, k, n), oracle, 1e-4)
    print(f"  split pair k={k} n={n} b={batch} {route} worst/bound={worst:.3g}", flush=True)
    assert route == "q4_mfma_pair_swiglu" and finite and ok
    # a row's sums are those of a call on its matrix (whose columns past 32 may take another route)
    (g, rg, _), (u, ru, _) = (run_matmul(Q4, w, x, k, n, batch) for w in (pg, pu))
    if rg == ru == SPLIT:
        expected = np.hstack([device_swiglu(np.ascontiguousarray(g[:32, c:c + 16384]), np.ascontiguousarray(u[:32, c:c + 16384]))
                              for c in range(0, n, 16384)])
        assert np.array_equal(y[:32].view(np.uint32), expected.view(np.uint32))
    else:
        assert (k, n) == (2048, 1000) and rg == ru == "q4_bdiag_gemv"
