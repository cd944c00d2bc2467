"""Decode attention by length: the kernels clamp and report lengths themselves, over chunk and
group edges, and calls of different head dims follow each other without seeing the other
layout's partials."""
import numpy as np
import pytest

from nimbleml_amd import _native as N
from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu


def want(q, k, v, lens, scale):
    q, k, v = (t.astype(np.float64) for t in (q, k, v))
    out = np.zeros_like(q)
    for b, n in enumerate(lens):
        s = np.einsum("hd,hkd->hk", q[b], k[b, :, :n]) / scale
        p = np.exp(s - s.max(-1, keepdims=True))
        out[b] = np.einsum("hk,hkd->hd", p / p.sum(-1, keepdims=True), v[b, :, :n])
    return out


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_head_dims_in_turn_at_edge_lengths(dtype):
    r = np.random.RandomState(3)
    lens = np.array([1, 63, 64, 65, 255, 256, 257, 700], np.int32)
    for dk in (40, 64, 8, 128, 200, 32, 256, 64):
        q = r.randn(8, 2, dk).astype(dtype)
        k, v = (r.randn(8, 2, 700, dk).astype(dtype) for _ in range(2))
        got = K.decode_attention(q, k, v, lens, float(np.sqrt(dk))).numpy().reshape(8, 2, dk)
        # fp16: scores below 8 rounded twice and their exponentials, values below 4; the output
        tol = 4 * (2 * 8 * 2.0**-11 + 2 * 2.0**-11) if dtype == np.float16 else 2e-5
        assert np.abs(got - want(q, k, v, lens, np.sqrt(dk))).max() <= tol, dk


@pytest.mark.parametrize("dk", [24, 64])
def test_lengths_outside_the_cache_are_clamped_and_reported(dk):
    r = np.random.RandomState(4)
    q = r.randn(3, 2, dk).astype(np.float32)
    k, v = (r.randn(3, 2, 130, dk).astype(np.float32) for _ in range(2))
    dev = [N.DeviceArray.from_host(t) for t in (q, k, v)]

    def run(lens):
        ln = N.DeviceArray.from_host(np.array(lens, np.int32))
        out, err = N.DeviceArray.from_host(np.zeros_like(q)), N.DeviceArray.from_host(np.zeros(1, np.int32))
        N.check(N.lib.nml_decode_attention_device(*(d.ptr for d in dev), ln.ptr, out.ptr, 3, 2, 130, dk,
                                                  float(np.sqrt(dk)), err.ptr, 0))
        return out.numpy(), int(err.numpy()[0])

    inside, none = run([1, 130, 130])
    clamped, told = run([0, 131, 2**31 - 1])
    assert none == 0 and told == 1
    assert np.array_equal(inside, clamped)
