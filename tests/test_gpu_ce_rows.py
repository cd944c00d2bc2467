"""The cross-entropy of logit rows held in registers: vocabularies at the edges of a thread's
chunks and past them, ignored labels; and the training step whose backward uses the forward's
logits and, the second time, forms them again."""
import ctypes as C

import numpy as np
import pytest

from nimbleml_amd import _native as N
from nimbleml_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("vocab", [3, 8, 1023, 1024, 4096, 4104, 8200, 16392, 32768, 32776, 65544])
def test_loss_over_vocab_edges(vocab, dtype):
    r = np.random.RandomState(vocab)
    h = r.randn(5, 64).astype(dtype)
    w = (r.randn(vocab, 64) * 0.1).astype(dtype)
    lab = r.randint(0, vocab, 5)
    lab[3] = 1
    x = h.astype(np.float64) @ w.astype(np.float64).T
    lse = np.log(np.exp(x - x.max(-1, keepdims=True)).sum(-1)) + x.max(-1)
    row = lse - x[np.arange(5), lab]
    # fp16: the logits (below 4) and the shifted exponents rounded to 11 bits
    tol = 4 * 2.0**-10 if dtype == np.float16 else 1e-5
    assert abs(K.fused_tied_crossentropy_forward(h, w, lab) - row.mean()) <= tol
    keep = lab != 1
    if keep.any():
        got = K.fused_tied_crossentropy_forward(h, w, lab, ignore_index=1)
        assert abs(got - row[keep].mean()) <= tol


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_second_backward_of_a_loss_equals_the_first(dtype):
    import nimbleml_amd as nm
    from oracle.weights import TINY, make_weights, random_ids

    cfg = TINY
    w = make_weights(cfg, seed=3, dtype=dtype, rich=True)
    m = nm.GPT.from_arrays(w, cfg.vocab_size, cfg.d_model, cfg.num_heads, cfg.num_layers,
                           cfg.max_seq_len, dtype=dtype)
    ids, lab = random_ids((2, 9), cfg.vocab_size, seed=5), random_ids((2, 9), cfg.vocab_size, seed=6)
    h, loss = m._device_model(), C.c_double()
    dids, dlab = N.DeviceArray.from_host(ids), N.DeviceArray.from_host(lab)
    head = np.ascontiguousarray(w["token_emb.weights"])

    def loss_train():
        N.check(N.lib.nml_model_loss_train(h, dids.ptr, dlab.ptr, 2, 9, 0, 0, C.byref(loss)))

    def set_head(scale):
        arr = np.ascontiguousarray(head * np.asarray(scale, dtype))
        N.check(N.lib.nml_model_set_param(h, N.P_TOKEN_EMB, 0, arr.ctypes.data, arr.nbytes))

    def backward():
        N.check(N.lib.nml_model_zero_grad(h))
        N.check(N.lib.nml_model_backward(h, 1.0))
        return [m._grad_array(k, 0, m._device_shape(k))
                for k in (N.P_TOKEN_EMB, N.P_LN_F, N.P_WQKV, N.P_W1, N.P_B2)]

    loss_train()
    first, second = backward(), backward()
    for x, y in zip(first, second):
        assert np.abs(x).max() > 0 and np.array_equal(x, y)
    # another head uploaded after the loss: its logits' gradient, in the first backward too
    set_head(2)
    changed = backward()
    assert not np.array_equal(changed[0], first[0])
    set_head(1)
    loss_train()
    set_head(2)
    for x, y in zip(backward(), changed):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("vocab,d", [(512, 64), (20000, 128)])
def test_head_written_through_an_earlier_pointer(vocab, d, dtype):
    """Between a loss and its backward the head changes in one element, through a pointer taken
    before the loss: the gradients are those of a backward that forms the logits itself."""
    import nimbleml_amd as nm
    from oracle.weights import GPTConfig, make_weights, random_ids

    cfg = GPTConfig(vocab, d, 4, 1, 16)
    w = make_weights(cfg, seed=3, dtype=dtype, rich=True)
    m = nm.GPT.from_arrays(w, cfg.vocab_size, cfg.d_model, cfg.num_heads, cfg.num_layers,
                           cfg.max_seq_len, dtype=dtype)
    ids, lab = random_ids((2, 9), vocab, seed=5), random_ids((2, 9), vocab, seed=6)
    h, loss, ptr = m._device_model(), C.c_double(), C.c_void_p()
    dids, dlab = N.DeviceArray.from_host(ids), N.DeviceArray.from_host(lab)
    head = np.ascontiguousarray(w["token_emb.weights"])
    other = head.copy()
    other[-1, -1] += np.asarray(4, dtype)

    def backward():
        N.check(N.lib.nml_model_zero_grad(h))
        N.check(N.lib.nml_model_backward(h, 1.0))
        return [m._grad_array(k, 0, m._device_shape(k)) for k in (N.P_TOKEN_EMB, N.P_LN_F, N.P_W1)]

    def loss_train():
        N.check(N.lib.nml_model_loss_train(h, dids.ptr, dlab.ptr, 2, 9, 0, 0, C.byref(loss)))

    loss_train()
    plain = backward()
    N.check(N.lib.nml_model_set_param(h, N.P_TOKEN_EMB, 0, other.ctypes.data, other.nbytes))
    want = backward()  # of the first loss, with the other head
    assert not np.array_equal(want[0], plain[0])
    N.check(N.lib.nml_model_set_param(h, N.P_TOKEN_EMB, 0, head.ctypes.data, head.nbytes))
    N.check(N.lib.nml_model_param_ptr(h, N.P_TOKEN_EMB, 0, C.byref(ptr)))
    loss_train()
    N.check(N.lib.nml_memcpy_h2d(ptr, other.ctypes.data, other.nbytes))
    for x, y in zip(backward(), want):
        assert np.array_equal(x, y)
    N.check(N.lib.nml_memcpy_h2d(ptr, head.ctypes.data, head.nbytes))
    loss_train()
    for x, y in zip(backward(), plain):
        assert np.array_equal(x, y)


def allocate(size):
    """A device block of that many bytes, or None."""
    p = C.c_void_p()
    return p.value if N.lib.nml_malloc(size, C.byref(p)) == 0 else None


def fill_memory(left):
    """Blocks that take the device's memory but for `left` bytes."""
    spare, blocks, size = allocate(left), [], 1 << 36
    while size >= 1 << 24:
        block = allocate(size)
        if block is None:
            size //= 2
        else:
            blocks.append(block)
    N.check(N.lib.nml_free(spare))
    x = N.DeviceArray.from_host(np.zeros(8, np.float32))
    N.lib.nml_gelu_forward_device(x.ptr, x.ptr, None, 8, N.F32)  # takes the last allocation's error
    return blocks


def release(blocks):
    for p in blocks:
        N.check(N.lib.nml_free(p))


@pytest.mark.parametrize("left", [48 << 20, 4 << 30])
def test_kept_logits_give_way(left):
    """With less memory left after the loss than the backward's scratch, the logits kept for it
    make the room; with little left before the loss, none are kept."""
    import nimbleml_amd as nm
    from oracle.weights import GPTConfig, make_weights, random_ids

    cfg, rows, seq = GPTConfig(50000, 512, 4, 1, 512), 8, 512
    w = make_weights(cfg, seed=3, dtype=np.float32)
    ids, lab = (random_ids((rows, seq), cfg.vocab_size, seed=s) for s in (5, 6))
    logits = rows * seq * cfg.vocab_size * 4  # 819 MB; half of it at a time without keeping them
    early = left > logits
    got = []
    for tight in (False, True):
        m = nm.GPT.from_arrays(w, cfg.vocab_size, cfg.d_model, cfg.num_heads, cfg.num_layers, cfg.max_seq_len,
                               dtype=np.float32)
        h, loss = m._device_model(), C.c_double()
        dids, dlab = N.DeviceArray.from_host(ids), N.DeviceArray.from_host(lab)
        N.check(N.lib.nml_model_zero_grad(h))
        blocks = fill_memory(left) if tight and early else []
        N.check(N.lib.nml_model_loss_train(h, dids.ptr, dlab.ptr, rows, seq, 0, 0, C.byref(loss)))
        if tight and early:  # the activations are 140 MB
            probe = allocate(left - 140 * 2**20 - logits * 3 // 4)
            assert probe is not None
            release([probe])
        elif tight:
            blocks = fill_memory(left)
        try:
            N.check(N.lib.nml_model_backward(h, 1.0))
        finally:
            release(blocks)
        got.append([m._grad_array(k, 0, m._device_shape(k)) for k in (N.P_TOKEN_EMB, N.P_LN_F, N.P_WQKV, N.P_B2)])
        del m
    for x, y in zip(*got):  # (a weight gradient over two chunks sums in another order)
        assert np.abs(x - y).max() <= 1e-5 * np.abs(x).max()
