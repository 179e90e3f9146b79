"""Backward's tiled products where their tiles and row packing change: the
head's packed target rows (gemm_mfma.hip's transposed operands, real
gradients), and the attention heads' products at the widths where the row
kernel takes another number of values per lane, against the CPU oracle.

Bar: within 1e-11 of the largest element, as in test_gpu_train.py (the
products sum in another order; the weights are scaled so that every gradient
stays near 1)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import rustcrates_amd as ra

pytestmark = pytest.mark.gpu

TOL = 1e-11


def c(r, *shape):
    return r.standard_normal(shape) + 1j * r.standard_normal(shape)


def far(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


# one target; a tile of target rows and one more; every row but the last; odd vocabularies and widths
@pytest.mark.parametrize("V,d,B,S,T", [(70, 8, 1, 2, 1), (129, 66, 5, 14, 13), (64, 64, 8, 9, 8), (1000, 20, 3, 40, 7),
                                       (9000, 7, 2, 70, 65)])
def test_head_gradients_and_update(V, d, B, S, T):
    r = np.random.default_rng(V + d)
    table, w, b = c(r, V, d), 0.2 * c(r, d, V), 0.1 * c(r, V)
    ids = r.integers(2, V, (B, S)).astype(np.uint32)
    targets = r.integers(2, V, (B, T)).astype(np.uint32)
    targets[0, 0] = 1  # PAD: its row has no target
    with ra.Network(0) as net:
        net.add_embedding(V, d, table)
        net.add_linear(d, V, w, b)
        net.add_softmax(ra.TRAINING)
        P, _ = net.predict(ids, forward_only=False)
        dx = net.backward_head(targets, update=True, learning_rate=0.01, time_step=1)
        w1, b1 = net.get_tensor(1, 0, d * V).reshape(d, V), net.get_tensor(1, 4, V)
    if T == 1:  # the only target is PAD: no gradient, nothing moves
        assert np.array_equal(w1, w) and np.array_equal(b1, b) and not dx.any()
        return
    dW, db, want = oracle.linear_backward(table[ids], oracle.softmax_backward(P, targets), w)
    zero = lambda *s: np.zeros(s, np.complex128)  # noqa: E731
    wo, bo = oracle.linear_update(w, b, dW, db, B, [zero(d, V), zero(d, V), zero(V), zero(V)], True, 0.01, 1)
    # the moves are at least 1e-6 of the weights they are subtracted from: eps / 1e-6
    assert far(dx, want) < TOL and far(w1 - w, wo - w) < 1e-9 and far(b1 - b, bo - b) < 1e-9


def test_rows_without_a_target_still_poison_their_weights():
    """An infinite input in a row without a target meets a zero gradient: NaN,
    which the update leaves out (linear_layer.rs:159-174)."""
    V, d, B, S, T = 90, 6, 2, 10, 3
    r = np.random.default_rng(1)
    table, w = c(r, V, d), 0.2 * c(r, d, V)
    table[5, 2] = complex(np.inf, 0.0)
    ids = r.integers(6, V, (B, S)).astype(np.uint32)
    ids[1, S - 1] = 5  # the last row predicts nothing
    targets = r.integers(6, V, (B, T)).astype(np.uint32)
    with ra.Network(0) as net:
        net.add_embedding(V, d, table)
        net.add_linear(d, V, w, np.zeros(V, np.complex128))
        net.add_softmax(ra.TRAINING)
        net.predict(ids, forward_only=False, want_output=False)
        net.backward_head(targets, update=True, learning_rate=0.5, time_step=1, want_grad_input=False)
        w1 = net.get_tensor(1, 0, d * V).reshape(d, V)
    assert np.array_equal(w1[2], w[2])
    assert all(np.all(w1[j] != w[j]) for j in range(d) if j != 2)


@pytest.mark.parametrize("S,d,H,norm", [(65, 16, 2, True), (129, 48, 2, False), (130, 20, 1, True), (513, 8, 2, True)])
def test_attention_input_gradient(S, d, H, norm):
    V, B, T = 70, 2, S // 2
    r = np.random.default_rng(S)
    table, wv = c(r, V, d), 0.1 * c(r, d, V)
    q, k, v = (0.3 * c(r, H, d, d // H) for _ in range(3))
    bias = 0.3 * c(r, H, S, S)
    one, nil = np.ones(d, np.complex128), np.zeros(d, np.complex128)
    ids = r.integers(2, V, (B, S)).astype(np.uint32)
    targets = r.integers(2, V, (B, T)).astype(np.uint32)
    lens = np.array([S, S - 3], np.uint32)

    def build(net):
        net.add_embedding(V, d, table)
        if norm:
            net.add_norm(d, 1e-5, one, nil)
        net.add_self_attention(H, d, S, 1e-12, q, k, v, bias, one, nil)
        net.add_linear(d, V, wv, np.zeros(V, np.complex128))
        net.add_softmax(ra.TRAINING)
        return net

    g, o = build(ra.Network(0)), build(oracle.Network())
    g.predict(ids, lens=lens, forward_only=False, want_output=False)
    dx = g.backward(targets, layers=2, update=False)
    g.close()
    P, mask = o.predict(ids, lens=lens, forward_only=False)
    x = table[ids] * mask[:, :, None]
    if norm:
        x = o.forward_layers(1, 2, x, mask=mask, forward_only=False)
    at = 2 if norm else 1
    y = o.forward_layers(at, at + 1, x, mask=mask, forward_only=False)
    o.close()
    gr = oracle.linear_backward(y, oracle.softmax_backward(P, targets), wv)[2]
    want = oracle.self_attention_backward(x, mask, q, k, v, bias, one, nil, gr)[0]
    assert far(dx, want) < TOL


def test_second_backward_reads_the_updated_weights():
    """The forward pass leaves a FeedForward's products for backward; after an
    update they are formed again from the layer's kept input."""
    V, d, F, B, S, T = 60, 8, 80, 2, 40, 9
    r = np.random.default_rng(5)
    table, w1, b1, w2, b2, wv = c(r, V, d), 0.3 * c(r, d, F), 0.1 * c(r, F), 0.2 * c(r, F, d), 0.1 * c(r, d), 0.1 * c(r, d, V)
    ids = r.integers(2, V, (B, S)).astype(np.uint32)
    targets = r.integers(2, V, (B, T)).astype(np.uint32)
    with ra.Network(0) as net:
        net.add_embedding(V, d, table)
        net.add_feed_forward(d, F, w1, b1, w2, b2)
        net.add_linear(d, V, wv, np.zeros(V, np.complex128))
        net.add_softmax(ra.TRAINING)
        P, mask = net.predict(ids, forward_only=False)
        net.backward(targets, layers=2, update=True, learning_rate=0.5, time_step=1, want_grad_input=False)
        dx = net.backward(targets, layers=2, update=False)
        n1, n2, nv = (net.get_tensor(1, 0, d * F).reshape(d, F), net.get_tensor(1, 1, F * d).reshape(F, d),
                      net.get_tensor(2, 0, d * V).reshape(d, V))
        nb = net.get_tensor(1, 4, F)
    assert far(n1, w1) > 1e-4
    x = table[ids]
    gelu = np.vectorize(lambda z: oracle.gelu(z)[0])
    head = gelu(x @ w1 + b1) @ w2 + b2  # the head's input is the forward pass's
    gr = oracle.linear_backward(head, oracle.softmax_backward(P, targets), nv)[2]
    z = x @ n1 + nb
    dh = oracle.linear_backward_c(gelu(z), gr, n2)[2]
    assert far(dx, oracle.dense_backward(x, z, dh, mask, n1)[2]) < TOL


@pytest.mark.parametrize("bad", [complex(np.inf, 1.0), complex(0.5, -np.inf), complex(np.nan, 1.0), complex(1.0, np.nan)])
def test_a_zero_gradient_row_meets_non_finite_head_weights(bad):
    """The rows without a target have a zero gradient; times a weight that is
    not finite, each of the four real products' sums is NaN."""
    V, d, B, S, T = 90, 6, 2, 10, 3
    r = np.random.default_rng(2)
    table, w = c(r, V, d), 0.2 * c(r, d, V)
    w[2, 71] = bad
    ids, targets = r.integers(2, V, (B, S)).astype(np.uint32), r.integers(2, V, (B, T)).astype(np.uint32)
    with ra.Network(0) as net:
        net.add_embedding(V, d, table)
        net.add_linear(d, V, w, np.zeros(V, np.complex128))
        net.add_softmax(ra.TRAINING)
        net.predict(ids, forward_only=False, want_output=False)
        dx = net.backward_head(targets, update=False)
    zero = np.ones(S, bool)
    zero[S - T - 1:S - 1] = False  # the rows that predict a target
    rest = [j for j in range(d) if j != 2]
    assert np.isnan(dx[:, zero, 2].real).all() and np.isnan(dx[:, zero, 2].imag).all()
    assert not dx[:, zero][:, :, rest].any()
