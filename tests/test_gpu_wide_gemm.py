"""GPU parity of the wide Q4_0 prefill tiles (256 and 128 activation rows x 256
weight rows, forced by KUNLUN_GEMM_TILE=256x64 and 128x64): one and several
weight super-stages, partial row and column tiles, the gate/up pair, subnormal
block scales (the F32 correction) and extreme rows. Bound as for the other
GEMM tiles: 2e-3 * ||x_b|| * ||w_r|| per element.
"""
import numpy as np
import pytest

import kunlunk200_lib_amd as kl
from gpu_util import run_matmul, weight_payload
from test_gpu_decode_edges import gemm_bound_ok, q4_sparse_subnormal, q4_subnormal
from test_gpu_gemm import check_gemm, gaussian
from test_gpu_swiglu import check_pair, run_pair

pytestmark = pytest.mark.gpu

Q4 = kl.WeightType.q4_0
WIDE = ["256x64", "128x64"]


@pytest.mark.parametrize("tile", WIDE)
@pytest.mark.parametrize("k,n,batch", [(256, 64, 64), (512, 700, 200), (768, 257, 129), (4096, 300, 513), (1024, 1, 256)])
def test_wide_tiles(gpu, oracle, knobs, tile, k, n, batch):
    knobs("KUNLUN_GEMM_TILE", tile)
    w = gaussian((n, k), 0.02, k + n)
    x = gaussian((batch, k), 1.0, k + n + 1)
    x[3] *= 1e6
    x[7] *= 1e-30
    payload, dec = weight_payload(Q4, w, oracle)
    y, route, guard_ok = run_matmul(Q4, payload, x, k, n, batch)
    finite, ok, _ = check_gemm(y, oracle.gold(dec, x, threads=16), dec, x)
    assert route == "q4_gemm_mfma" and guard_ok and finite and ok


@pytest.mark.parametrize("tile", WIDE)
@pytest.mark.parametrize("k,n,batch", [(512, 300, 130), (4096, 129, 300)])
def test_wide_pair(gpu, oracle, knobs, tile, k, n, batch):
    knobs("KUNLUN_GEMM_TILE", tile)
    x = gaussian((batch, k), 1.0, 3)
    pg, dg = weight_payload(Q4, gaussian((n, k), 0.02, 1), oracle)
    pu, du = weight_payload(Q4, gaussian((n, k), 0.02, 2), oracle)
    y, route = run_pair(Q4, pg, pu, x, k, n, batch)
    finite, ok, worst = check_pair(y, x, dg, du, oracle, 2e-3)
    assert route == "q4_gemm_swiglu_mfma" and finite and ok, worst


@pytest.mark.parametrize("tile", WIDE)
@pytest.mark.parametrize("sparse", [False, True], ids=["mixed", "sparse"])
def test_wide_subnormal_scales(gpu, oracle, knobs, tile, sparse):
    knobs("KUNLUN_GEMM_TILE", tile)
    k, n, batch = (4096, 700, 200) if sparse else (512, 200, 160)
    q4 = q4_sparse_subnormal(k, n, 97) if sparse else q4_subnormal(k, n, 91, True, tiny=True)
    dec = oracle.q4_decode(q4, k, n)
    x = np.random.default_rng(98).standard_normal((batch, k)).astype(np.float32)
    y, route, guard_ok = run_matmul(Q4, q4, x, k, n, batch)
    assert route == "q4_gemm_mfma" and guard_ok and np.all(np.isfinite(y))
    ok, ratio = gemm_bound_ok(y, oracle.gold(dec, x, threads=16), dec, x, 2e-3)
    assert ok, f"tile {tile}: error {ratio:.3g} x the bound"


@pytest.mark.parametrize("tile", WIDE)
def test_wide_pair_subnormal_scales(gpu, oracle, knobs, tile):
    knobs("KUNLUN_GEMM_TILE", tile)
    k, n, batch = 1024, 150, 140
    pg, pu = q4_sparse_subnormal(k, n, 11), q4_sparse_subnormal(k, n, 12)
    x = np.random.default_rng(13).standard_normal((batch, k)).astype(np.float32)
    y, route = run_pair(Q4, pg, pu, x, k, n, batch)
    finite, ok, worst = check_pair(y, x, oracle.q4_decode(pg, k, n), oracle.q4_decode(pu, k, n), oracle, 2e-3)
    assert route == "q4_gemm_swiglu_mfma" and finite and ok, worst
