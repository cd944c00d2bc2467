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


@pytest.mark.parametrize("dk", [16, 32, 96, 128])
def test_probability_of_a_large_score(dk):
    """One key per row has all the weight, its score far from zero: P is exp(s - lse) = 1 to the
    bit, so dV is dO there (lse·log2(e) rounded by itself put P off by 2^-24·|lse|)."""
    seq, scale = 70, 4.0
    q, k = np.zeros((1, seq, dk), np.float32), np.zeros((1, seq, dk), np.float32)
    k[0, :, 0], k[0, :, 1], k[0, 0, 0] = -64.0, 3.0, 64.0  # key 0: 81 more than all the others
    q[0, :, 0], q[0, :, 1] = 5.0, np.arange(seq) % 8 + 1.0
    do = np.random.RandomState(dk).randn(1, seq, dk).astype(np.float32)
    v = np.ones((1, seq, dk), np.float32)
    _, m, lsum = K.flash_sdpa_forward(q, k, v, scale)
    got = K.flash_sdpa_backward(do, q, k, v, m, lsum, scale)[2].numpy()
    assert (lsum.numpy() == 1).all() and (m.numpy() > 75).all()
    # the sum of dO over the rows, in float32 in some order: 70 terms below 5
    assert np.abs(got[0, 0] - do[0].astype(np.float64).sum(0)).max() <= 70 * 2.0**-24 * np.abs(do).sum(1).max()
    one = K.flash_sdpa_forward(q[:, :1], k[:, :1], v[:, :1], scale)
    alone = K.flash_sdpa_backward(do[:, :1], q[:, :1], k[:, :1], v[:, :1], one[1], one[2], scale)[2].numpy()
    assert np.array_equal(alone, do[:, :1])


@pytest.mark.parametrize("dk", [8, 32, 48, 96, 128])
@pytest.mark.parametrize("seq", [1, 65, 130])
def test_fp16_backward_head_dims(gpu, seq, dk):
    """The fp16 backward by itself: a causal attention layer with identity projections, whose
    input gradient is dQ + dK + dV. Scores below 4 in two fp16 roundings put P off by 2^-8 at
    most, the output and the three gradients are rounded once (2^-11 each)."""
    import nimbleml_amd as nm
    from oracle import gpt_ref as R
    from oracle import grad_ref as G
    from oracle.weights import GPTConfig, make_weights

    cfg = GPTConfig(64, 2 * dk, 2, 1, 256)
    w = {n: a.astype(np.float16) for n, a in make_weights(cfg, seed=1, dtype=np.float32, rich=True).items()}
    pm = "blocks.layers.0.mha."
    for n in ("W_q", "W_k", "W_v", "W_o"):
        w[pm + n + ".weights"] = np.eye(2 * dk, dtype=np.float16)
        w[pm + n + ".biases"] = np.zeros_like(w[pm + n + ".biases"])
    r = np.random.RandomState(seq + dk)
    x, dout = ((0.5 * r.randn(2, seq, 2 * dk)).astype(np.float16) for _ in range(2))
    old = nm.np_backend.dtype
    nm.set_dtype("float16")
    try:
        mha = nm.GPT.from_arrays(w, 64, 2 * dk, 2, 1, 256, dtype=np.float16)._block_list[0].mha
        mask = R.causal_mask(seq, np.float16)
        xt = nm.Tensor(x, x.shape, requires_grad=True)
        mha(xt, nm.Tensor(mask, mask.shape)).backward(dout)
        got = np.asarray(xt.grad, np.float64).reshape(x.shape)
    finally:
        nm.set_dtype(np.dtype(old).name)
    want = G.mha_vjp({n: a.astype(np.float64) for n, a in w.items()}, pm, x.astype(np.float64),
                     dout.astype(np.float64), 2, R.causal_mask(seq, np.float64))[1]
    assert np.abs(got - want).max() <= (2.0**-8 + 4 * 2.0**-11) * np.abs(want).max()
