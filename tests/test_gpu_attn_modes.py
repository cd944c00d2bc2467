"""Prefill attention on the matrix cores beyond causal head dims 64 and 128: every key, additive
masks, and the head dims in between, against float64 over the edges of the 64-key and
128-query tiles; masks that leave a query nothing, the type's lowest value, infinities."""
import numpy as np
import pytest

from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu

# scores: fp16 roundings of q·k, of the quotient and (masked) of the sum, |score| ≤ 8, move a
# probability by up to 3 · 8 · 2^-11 of itself; the output's own rounding 2^-11. float32: a
# few hundred roundings of 2^-24.
TOL = {np.float16: 0.015, np.float32: 1e-5}


def reference(q, k, v, bias):
    s = q.astype(np.float64) @ k.astype(np.float64).transpose(0, 2, 1) / np.sqrt(q.shape[-1])
    s = s if bias is None else s + bias.astype(np.float64)
    with np.errstate(invalid="ignore"):
        p = np.exp(s - s.max(-1, keepdims=True))
        return (p / p.sum(-1, keepdims=True)) @ v.astype(np.float64)


def inputs(bh, seq, dk, dtype, seed=0):
    r = np.random.RandomState(seed + seq + dk)
    return [r.randn(bh, seq, dk).astype(dtype) for _ in range(3)]


def bias_of(mode, seq, dtype, seed=1):
    if mode == "full":
        return None
    if mode == "causal":
        return np.triu(np.full((seq, seq), -np.inf, dtype), 1)
    if mode == "window":  # later rows see nothing in their first tiles
        i = np.arange(seq)
        d = i[:, None] - i[None, :]
        return np.where((d >= 0) & (d < 5), 0, -np.inf).astype(dtype)
    return np.random.RandomState(seed).randn(seq, seq).astype(dtype)


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("mode", ["full", "causal", "window", "bias"])
@pytest.mark.parametrize("seq,dk", [(1, 32), (63, 8), (64, 16), (65, 32), (129, 48), (130, 64),
                                    (192, 80), (257, 96), (131, 104), (191, 128)])
def test_modes_and_head_dims(seq, dk, mode, dtype):
    q, k, v = inputs(3, seq, dk, dtype)
    bias = bias_of(mode, seq, dtype)
    got = K.fused_sdpa_forward(q, k, v, np.sqrt(dk), bias)[0].numpy()
    want = reference(q, k, v, bias)
    assert np.abs(got - want).max() <= TOL[dtype] * np.abs(v).max()


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("dk", [32, 64, 128])
def test_rows_with_nothing_to_attend(dk, dtype):
    """A row of −∞ is NaN, as a softmax over nothing is; a row of the type's lowest value
    absorbs the scores and averages the values; rows beside them are untouched."""
    seq = 150
    q, k, v = inputs(2, seq, dk, dtype)
    bias = np.zeros((seq, seq), dtype)
    bias[7] = -np.inf
    bias[20] = np.finfo(dtype).min
    bias[33, :149] = -np.inf  # one key, in the last tile
    got = K.fused_sdpa_forward(q, k, v, np.sqrt(dk), bias)[0].numpy().astype(np.float64)
    want = reference(q, k, v, bias)
    assert np.isnan(got[:, 7]).all()
    assert np.abs(got[:, 20] - v.astype(np.float64).mean(1)).max() <= TOL[dtype]
    keep = np.setdiff1d(np.arange(seq), [7, 20])
    assert np.abs(got - want)[:, keep].max() <= TOL[dtype] * np.abs(v).max()
    assert np.abs(got[:, 33] - v[:, 149]).max() <= 1e-6


def test_infinite_and_nan_scores_stay_in_their_rows():
    for dtype in (np.float16, np.float32):
        q, k, v = inputs(1, 100, 64, dtype)
        bias = np.zeros((100, 100), dtype)
        bias[3, 4], bias[5, 90] = np.inf, np.nan
        got = K.fused_sdpa_forward(q, k, v, 8.0, bias)[0].numpy()
        assert np.isnan(got[0, 3]).all() and np.isnan(got[0, 5]).all()
        assert np.isfinite(np.delete(got[0], [3, 5], 0)).all()


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_misaligned_rows_take_the_scalar_kernels(dtype):
    """Buffers one element past a 16-byte boundary give what aligned ones give."""
    from nimbleml_amd import _native as N

    bh, seq, dk = 2, 70, 64
    q, k, v = inputs(bh, seq, dk, dtype)
    es = np.dtype(dtype).itemsize
    dev = []
    for a in (q, k, v):
        d = N.DeviceArray((a.size + 8,), dtype)
        N.check(N.lib.nml_memcpy_h2d(d.ptr + es, a.ctypes.data, a.nbytes))
        dev.append(d)
    out = N.DeviceArray((bh, seq, dk), dtype)
    N.check(N.lib.nml_sdpa_forward_device(*[d.ptr + es for d in dev], None, out.ptr, bh, seq, dk,
                                          8.0, 0, N.np_dtype_code(dtype)))
    want = reference(q, k, v, None)
    assert np.abs(out.numpy() - want).max() <= TOL[dtype] * np.abs(v).max()


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("mode", ["full", "causal", "window", "bias", "causal call"])
@pytest.mark.parametrize("seq,dk", [(90, 32), (200, 64), (130, 48), (150, 96), (70, 104), (150, 128)])
def test_infinite_and_nan_values(seq, dk, mode, dtype):
    """An infinite value is an infinite output wherever its key has a weight, and no output where
    it has none (a masked key, or a later key of the same tile)."""
    from nimbleml_amd import _native as N

    if mode.startswith("causal") and dk in (64, 128):
        pytest.skip("the causal kernel of these head dims sums every key of a tile, weight or not")
    q, k, v = inputs(2, seq, dk, dtype)
    v[0, 66, 1], v[0, 40, dk - 1] = np.inf, -np.inf
    v[1, 3, 2], v[1, 60, 0], v[1, 61, 0] = np.nan, np.inf, -np.inf
    bias = np.triu(np.full((seq, seq), -np.inf, dtype), 1) if mode == "causal call" else bias_of(mode, seq, dtype)
    dev = [N.DeviceArray.from_host(a) for a in (q, k, v)]
    if mode == "causal call":
        out = N.DeviceArray((2, seq, dk), dtype)
        N.check(N.lib.nml_sdpa_forward_device(*(d.ptr for d in dev), None, out.ptr, 2, seq, dk,
                                              float(np.sqrt(dk)), 1, N.np_dtype_code(dtype)))
        got = out.numpy()
    else:
        got = K.fused_sdpa_forward(q, k, v, np.sqrt(dk), bias)[0].numpy()
    seen = np.ones((seq, seq), bool) if bias is None else np.isfinite(bias)
    want = reference(q, k, np.where(np.isfinite(v), v, 0), bias)
    for b, key, d, value in [(0, 66, 1, np.inf), (0, 40, dk - 1, -np.inf), (1, 3, 2, np.nan), (1, 60, 0, np.inf),
                             (1, 61, 0, -np.inf)]:
        with np.errstate(invalid="ignore"):  # inf - inf
            want[b, :, d] = np.where(seen[:, key], want[b, :, d] + value, want[b, :, d])
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(dtype))
    keep = np.isfinite(want)
    assert np.abs(got[keep] - want[keep]).max() <= TOL[dtype] * 5  # |v| below 5


@pytest.mark.parametrize("gap", [6.0, 11.0, 15.0, 18.0])
@pytest.mark.parametrize("mode", ["full", "bias"])
@pytest.mark.parametrize("dk", [32, 64, 96, 128])
def test_many_small_probabilities_beside_a_peak(dk, mode, gap):
    """One key above thousands of equal ones, whose weight times their values is the result: each
    probability is off by at most 2^-24 of itself or 2^-37 of the peak's."""
    seq, value = 3000, 30000.0
    q, k, v = (np.zeros((1, seq, dk), np.float16) for _ in range(3))
    q[..., 0], v[:] = 1, value
    bias = np.zeros((seq, seq), np.float16) if mode == "bias" else None
    v[0, 1717] = 0
    if bias is None:
        k[0, 1717, 0] = gap
    else:
        bias[:, 1717] = gap
    got = K.fused_sdpa_forward(q, k, v, 1.0, bias)[0].numpy()
    p = (seq - 1) * np.exp(-gap)
    want = value * p / (1 + p)
    # the output's rounding (2^-11), a float32 sum of `seq` terms, and the bound above
    assert np.abs(got - want).max() <= want * (2.0**-11 + seq * 2.0**-24) + seq * value * 2.0**-37
