"""SoftmaxLayer's rows at the widths where its kernel changes (values per
thread, threads per row, the three-pass form), padded rows included, against
numpy on the same real logits.

Bound: the logits' own rounding (K = 4 terms of at most a few units) enters
the exponent, so a probability is within about 40 eps of numpy's relatively;
the sums of V terms add at most log2(V) + 8 roundings on top: 1e-13 covers both.
"""
from __future__ import annotations

import numpy as np
import pytest

import rustcrates_amd as ra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [3, 2048, 2049, 8192, 8193, 32768, 32769, 53248, 53249])
@pytest.mark.parametrize("mode", [ra.TRAINING, ra.PRODUCTION])
def test_softmax_rows(V, mode):
    d, B, S = 4, 2, 3
    r = np.random.default_rng(V)
    table = r.standard_normal((V, d)) + 1j * r.standard_normal((V, d))
    w = r.standard_normal((d, V)) + 1j * r.standard_normal((d, V))
    b = r.standard_normal(V) + 0j
    ids = np.array([[0, 2, V - 1], [2, 0, 1]], np.uint32)
    with ra.Network(0) as net:
        net.add_embedding(V, d, table)
        net.add_linear(d, V, w, b)
        net.add_softmax(mode)
        got, _ = net.predict(ids, lens=[3, 2], forward_only=False)
    x = table[ids]
    x[ids == 1] = 0
    lg = (x @ w + b).real
    e = np.exp(lg - lg.max(-1, keepdims=True))
    want = e / e.sum(-1, keepdims=True)
    live = np.array([[1, 1, 1], [1, 1, 0]]) if mode == ra.TRAINING else np.array([[0, 0, 1], [0, 0, 1]])
    want *= live[:, :, None]
    assert got.shape == want.shape
    assert np.max(np.abs(got - want) / np.where(want == 0, 1.0, want)) < 1e-13
