"""Top-p sampling from registers against a float64 walk: vocabularies at the edges of the
elements a thread holds, the draw at both ends of the kept set, and rows that the bins decline."""
import numpy as np
import pytest

from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu


def check(lg, top_k, top_p, u, temperature=0.8):
    """Every chosen token sits where u falls in the walk (models/generate.py:43-58; equal
    probabilities by descending index), its interval widened by what float32 probabilities
    (a few 2^-24 each, relative) move the running sums: 1e-5 of the mass."""
    got = K.sample_tokens(lg, temperature=temperature, top_k=top_k, top_p=top_p, uniforms=u)
    for b, row in enumerate(lg):
        x = row.astype(np.float32) / np.float32(temperature)
        if top_k and top_k < x.size:
            x = np.where(x < np.partition(x, -top_k)[-top_k], np.float32(-1e9), x)
        p = np.exp(x.astype(np.float64) - x.max())
        p /= p.sum()
        order = np.lexsort((np.arange(x.size), x))[::-1]
        cdf = np.cumsum(p[order])
        at = int(np.flatnonzero(order == got[b])[0])
        before, after = cdf[at] - p[order[at]], cdf[at]
        # the kept mass: everything up to top_p, at least the first; it may end one element
        # early or late
        ends = [cdf[max(0, e)] for e in (int(np.searchsorted(cdf, top_p + d, "right")) - 1
                                         for d in (-1e-5, 0.0, 1e-5))]
        assert any(before / e - 1e-5 <= u[b] <= after / e + 1e-5 for e in ends), (b, at, u[b])


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("vocab", [5, 1023, 1025, 4096, 4097, 16384, 16385, 32768, 32769, 50304, 51200, 51201])
@pytest.mark.parametrize("top_k,top_p", [(0, 0.9), (40, 0.95), (0, 0.05)])
def test_vocab_edges(vocab, top_k, top_p, dtype):
    r = np.random.RandomState(vocab + top_k)
    lg = (r.randn(6, vocab) * 2.5).astype(dtype)
    # (both ends of the kept set, and between)
    check(lg, top_k, top_p, np.array([1e-9, 0.1, 0.5, 0.9, 0.999, 1 - 1e-9]))


@pytest.mark.parametrize("scale", [0.0, 0.02, 30.0])
def test_flat_and_peaked_rows(scale):
    """Equal logits (every element in one bin: the general path), nearly equal ones, and a row
    whose first token alone exceeds top-p."""
    r = np.random.RandomState(5)
    lg = (r.randn(4, 4000) * scale).astype(np.float32)
    check(lg, 0, 0.9, np.array([0.03, 0.31, 0.62, 0.97]))


def test_masked_tokens():
    """Logits of −∞ (tokens ruled out) carry no mass."""
    r = np.random.RandomState(6)
    lg = (r.randn(4, 3000) * 2).astype(np.float32)
    lg[:, 7:2990] = -np.inf
    check(lg, 0, 0.9, np.array([0.03, 0.31, 0.62, 0.97]))
    check(lg, 5, 0.9, np.array([0.03, 0.31, 0.62, 0.97]))


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("vocab", [40, 1000, 1024, 3000])
@pytest.mark.parametrize("top_k", [0, 7])
def test_rows_without_probabilities(vocab, top_k, dtype):
    """Rows whose probabilities are NaN (a NaN or infinite logit, no finite logit) give the last
    token whatever the vocabulary, as a walk over one tied key does; a row beside them is its own."""
    r = np.random.RandomState(vocab)
    lg = r.randn(4, vocab).astype(dtype)
    lg[0, 5], lg[1, 6] = np.nan, np.inf
    lg[2] = -np.inf
    got = K.sample_tokens(lg, temperature=0.8, top_k=top_k, top_p=0.9, uniforms=np.full(4, 0.5))
    alone = K.sample_tokens(lg[3:], temperature=0.8, top_k=top_k, top_p=0.9, uniforms=np.full(1, 0.5))
    assert (got[:3] == vocab - 1).all(), got
    assert got[3] == alone[0]
