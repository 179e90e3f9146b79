"""What a network does where the device has no room: a request too large for
any GPU is an error and nothing else.

greedy_decoding of 2^20 rows of 2^31 ids asks for 2^54 bytes before it reads
its argument, so it is refused on every device without using any memory."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import rustcrates_amd as ra

pytestmark = pytest.mark.gpu


def ask_for_too_much(net):
    lg, ids = np.zeros(1), np.zeros(1, np.uint32)
    rc = net._lib.mitok_greedy_decoding(net._h, lg.ctypes.data_as(C.c_void_p), 2**20, 2**31,
                                        ids.ctypes.data_as(C.c_void_p))
    assert ra.ERRORS[rc] == "ERR_NOMEM"


def training_net(seed=3, V=70, d=16, H=2, F=48, S=33):
    net = ra.Network(0)
    net.add_embedding(V, d)
    net.add_norm(d, 1e-5)
    net.add_self_attention(H, d, S, 1e-12)
    net.add_feed_forward(d, F)
    net.add_linear(d, V)
    net.add_softmax(ra.TRAINING)
    net.init_seeded(seed)
    r = np.random.default_rng(seed)
    ids, targets = r.integers(2, V, (3, S)).astype(np.uint32), r.integers(2, V, (3, 9)).astype(np.uint32)
    return net, ids, np.array([S, S - 4, S], np.uint32), targets


def test_a_refused_allocation_leaves_no_error_behind():
    """The runtime keeps a failed allocation as the thread's last error until
    it is read; a later call must not take it for its own."""
    net, ids, lens, targets = training_net()
    with net:
        want, _ = net.predict(ids, lens=lens, forward_only=False)
        loss = net.cross_entropy_loss(targets)
        ask_for_too_much(net)
        assert net.cross_entropy_loss(targets) == loss
        ask_for_too_much(net)
        got, _ = net.predict(ids, lens=lens, forward_only=False)
    assert np.array_equal(got, want)


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # the library's runtime
    return free.value


def step(net, ids, lens, targets, before_backward=lambda: None):
    """One training step and a second backward under the new weights."""
    P, _ = net.predict(ids, lens=lens, forward_only=False)
    before_backward()
    g1 = net.backward(targets, layers=net.num_layers - 1, update=True, learning_rate=0.05, time_step=1)
    g2 = net.backward(targets, layers=4, update=False)
    return [P, g1, g2, net.get_tensor(2, 0, 16 * 16), net.get_tensor(3, 0, 16 * 48), net.get_tensor(4, 0, 16 * 70)]


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def test_backward_forms_products_that_were_not_kept():
    """Kept products, none kept, and kept ones given up before backward: the
    same kernels on the same rows, so the same bits."""
    runs = []
    for keep, give_up in ((True, False), (False, False), (True, True)):
        net, ids, lens, targets = training_net()
        with net:
            net.set_product_saving(keep)
            runs.append(step(net, ids, lens, targets, (lambda: ask_for_too_much(net)) if give_up else lambda: None))
    assert np.abs(runs[0][1]).max() > 0 and not np.array_equal(runs[0][1], runs[0][2])
    assert same(runs[0], runs[1]) and same(runs[0], runs[2])


def test_kept_products_give_way_to_another_allocation():
    net, ids, lens, targets = training_net(d=64, F=2048, S=400)
    held = ids.size * 16 * (2 * 2048 + 3 * 64)
    with net:
        P, _ = net.predict(ids, lens=lens, forward_only=False)
        before = free_bytes()
        ask_for_too_much(net)
        assert free_bytes() >= before + held // 2
        loss = net.cross_entropy_loss(targets)
        assert np.isfinite(loss.real)
        after, _ = net.predict(ids, lens=lens, forward_only=False)  # nothing took their place: kept again
        assert np.array_equal(after, P) and free_bytes() < before + held // 2
