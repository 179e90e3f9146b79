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
