"""GPU parity of native_q4_matmul above one column (int8 MFMA, the three digits
of up to 5 columns in one MFMA per block, a call's column groups in one launch
as long as it holds them): full and partial column groups, blocks that do not
fill the waves, one and several LDS chunks of activations, remainders of N,
unaligned F32 and F16 X, columns of very different size and non-finite
activations. Same bounds as the other
native Q4 tests: exact up to the activations' 23-bit block fixed point.
"""
import numpy as np
import pytest

import kunlunk200_lib_amd as kl
from test_gpu_native_q4 import NativeCase, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16,x_offset", [(False, 4), (True, 2)], ids=["f32", "f16"])
@pytest.mark.parametrize("k,n,batch", [(32, 1, 2), (96, 33, 5), (288, 64, 6), (4096, 40, 5), (4096, 100, 15), (5152, 31, 16),
                                       (2080, 65, 17), (16384, 32, 21), (1024, 31, 33), (11008, 70, 3)])
def test_native_columns(gpu, oracle, k, n, batch, f16, x_offset):
    case = NativeCase(oracle, k, n)
    x = np.random.default_rng(k + n + batch).standard_normal((batch, k)).astype(np.float32)
    x[1] *= 1e-3
    x[0, : k // 2] *= 200.0
    if f16:
        x = x.astype(np.float16).astype(np.float32)
    y, flag = case.run(kl.NativeQ4Workspace(), x, batch, f16=f16, x_offset=x_offset)
    assert not flag
    check(oracle, case, y, x)


@pytest.mark.parametrize("batch", [4, 16])
def test_native_columns_nonfinite(gpu, oracle, batch):
    k, n = 4096, 70
    case = NativeCase(oracle, k, n)
    x = np.random.default_rng(batch).standard_normal((batch, k)).astype(np.float32)
    x[1, 5], x[2, k - 1] = np.nan, np.inf
    y, _ = case.run(kl.NativeQ4Workspace(), x, batch)
    keep = np.delete(np.arange(batch), (1, 2))
    assert np.all(np.isnan(y[1:3]))
    check(oracle, case, y[keep], x[keep])


def test_native_more_columns_than_a_launch_holds(gpu, oracle):
    # 8 workgroups of 512 threads per 5 columns: more than 2^32 threads, in two launches
    k, n, batch = 32, 1, 5_300_000
    case = NativeCase(oracle, k, n)
    x = np.random.default_rng(3).standard_normal((1000, k)).astype(np.float16).astype(np.float32)
    small, _ = case.run(kl.NativeQ4Workspace(), x, 1000, f16=True)
    check(oracle, case, small, x)
    y, _ = case.run(kl.NativeQ4Workspace(), np.tile(x.astype(np.float16), (batch // 1000, 1)), batch, f16=True)
    assert np.array_equal(y.reshape(-1, 1000).view(np.uint32), np.broadcast_to(small.view(np.uint32).T, (batch // 1000, 1000)))
