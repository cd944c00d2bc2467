"""Projections of a few rows (csrc/ops_gemm.hip rows_kernel): every row count at which the
tiles or the division of K change, K at the edges of a load block and of the waves' shares,
narrow and odd outputs, all epilogues, against float64."""
import numpy as np
import pytest

from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu


def want(x, w, b, r, epi, dtype):
    y = x.astype(np.float64) @ w.astype(np.float64)
    if epi:
        y = y + b
    if epi == 2:
        y = 0.5 * y * (1 + np.tanh(0.7978845608028654 * (y + 0.044715 * y ** 3)))
    return y + r if epi == 3 else y


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("rows", [2, 3, 4, 5, 8, 9, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("n,k", [(1, 8), (17, 40), (1023, 264), (1024, 4096), (2056, 1032), (8200, 72)])
def test_rows_against_float64(rows, n, k, dtype):
    r = np.random.RandomState(rows * 7 + n + k)
    x, w = r.randn(rows, k).astype(dtype), (r.randn(k, n) / np.sqrt(k)).astype(dtype)
    b, res = r.randn(n).astype(dtype), r.randn(rows, n).astype(dtype)
    for epi in range(4):
        got = K.linear(x, w, b if epi else None, epilogue=epi, resid=res if epi == 3 else None).numpy()
        ref = want(x, w, b, res, epi, dtype)
        # fp16: three roundings of values below 8 (product, bias, residual or GELU); float32: the
        # sum's roundings, Σ|x||w| ≤ 4 and at most k / 16 + 32 additions, and the epilogue's
        tol = 3 * 8 * 2.0**-11 if dtype == np.float16 else (k / 16 + 40) * 2.0**-24 * 8
        assert np.abs(got - ref).max() <= tol, epi
