"""Causal attention backward on the matrix cores at head dims below the padded tiles (and one
that they do not take), at the edges of the 64-row tiles, against float64."""
import numpy as np
import pytest

from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk", [4, 8, 30, 32, 36, 64, 96, 100, 128])
@pytest.mark.parametrize("seq", [1, 63, 65, 130])
def test_flash_backward_head_dims(seq, dk):
    r = np.random.RandomState(seq + dk)
    q, k, v, do = (r.randn(3, seq, dk).astype(np.float32) for _ in range(4))
    scale = np.sqrt(dk)
    _, m, lsum = K.flash_sdpa_forward(q, k, v, scale)
    got = [g.numpy() for g in K.flash_sdpa_backward(do, q, k, v, m, lsum, scale)]
    q, k, v, do = (a.astype(np.float64) for a in (q, k, v, do))
    s = q @ k.transpose(0, 2, 1) / scale + np.triu(np.full((seq, seq), -np.inf), 1)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    dp = do @ v.transpose(0, 2, 1)
    ds = p * (dp - (dp * p).sum(-1, keepdims=True)) / scale
    for g, w in zip(got, (ds @ k, ds.transpose(0, 2, 1) @ q, p.transpose(0, 2, 1) @ do)):
        # float32 sums of at most 130 terms of |ds|, |p| ≤ 10 against operands below 5
        assert np.abs(g - w).max() <= 2e-5 * max(1.0, np.abs(w).max())
