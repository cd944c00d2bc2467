"""fp16 projections of few 64 × 64 tiles (csrc/ops_gemm.hip gemm_f16_t64_kernel): rows and
columns at the edges of a tile and of the rule, odd widths, K of fewer stages than the ring and
of many, with and without a half stage at the end, all epilogues, against float64."""
import numpy as np
import pytest

from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n", [(65, 1), (65, 64), (127, 72), (128, 1001), (200, 136), (255, 8192), (255, 8200),
                                    (256, 4096), (257, 1024), (1025, 960)])
@pytest.mark.parametrize("k", [256, 320, 384, 448, 512, 576, 2112])
def test_tiles_against_float64(rows, n, k):
    r = np.random.RandomState(rows + n + k)
    x, w = r.randn(rows, k).astype(np.float16), (r.randn(k, n) / np.sqrt(k)).astype(np.float16)
    b, res = r.randn(n).astype(np.float16), r.randn(rows, n).astype(np.float16)
    y = x.astype(np.float64) @ w.astype(np.float64)
    yb = y + b
    ref = [y, yb, 0.5 * yb * (1 + np.tanh(0.7978845608028654 * (yb + 0.044715 * yb ** 3))), yb + res]
    for epi in range(4):
        got = K.linear(x, w, b if epi else None, epilogue=epi, resid=res if epi == 3 else None).numpy()
        # three roundings (product, bias, residual or GELU) of values below 16, most below 8
        assert np.abs(got - ref[epi]).max() <= 3 * 16 * 2.0**-11 / 2, epi
