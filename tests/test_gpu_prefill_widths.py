"""The tiled prefill attention where its blocks change (32, 64 or 128 query
rows, one or two key groups, one head dim padded to the next built one), with
padded rows, against plain numpy in double precision.

Bound: a score is a real dot product of 2 dh terms, an output a sum of S
weighted values; the weights' errors are the scores' absolute ones, so 1e-12
of the largest output covers S up to a few hundred."""
from __future__ import annotations

import numpy as np
import pytest

import rustcrates_amd as ra

pytestmark = pytest.mark.gpu


def heads_output(x, wq, wk, wv, bias, mask):
    B, S, d = x.shape
    H, _, dh = wq.shape
    out = np.zeros((B, S, d), np.complex128)
    low = np.triu(np.ones((S, S), bool), 1)
    for b in range(B):
        for h in range(H):
            q, k, v = x[b] @ wq[h], x[b] @ wk[h], x[b] @ wv[h]
            s = (q @ k.T).real / (1e-8 + np.sqrt(dh)) + bias[h, :S, :S].real
            s[low] = -1e12
            p = np.exp(s - s.max(-1, keepdims=True))
            out[b, :, h * dh:(h + 1) * dh] = (p / p.sum(-1, keepdims=True)) @ v * mask[b][:, None]
    return out


# (B, S, H, dh): 32-row blocks with ragged ends, 64-row ones, 128-row ones; head dims between the built ones
@pytest.mark.parametrize("B,S,H,dh", [(1, 1, 2, 16), (2, 33, 2, 24), (1, 97, 1, 64), (64, 65, 2, 16), (70, 30, 4, 20),
                                      (130, 40, 4, 8), (40, 129, 5, 40), (2, 70, 2, 100), (1, 31, 1, 128),
                                      (130, 40, 4, 20), (43, 150, 4, 32)])
def test_prefill_attention_blocks(B, S, H, dh):
    d = H * dh
    r = np.random.default_rng(S * dh)
    c = lambda *s: r.standard_normal(s) + 1j * r.standard_normal(s)  # noqa: E731
    wq, wk, wv = (c(H, d, dh) / np.sqrt(2 * d) for _ in range(3))
    bias, x = 0.3 * c(H, S + 2, S + 2), c(B, S, d)
    lens = np.full(B, S)
    lens[-1] = max(1, S - 5)
    mask = (np.arange(S)[None, :] < lens[:, None]).astype(np.uint32)
    one, nil = np.ones(d, np.complex128), np.zeros(d, np.complex128)
    with ra.Network(0) as net:
        net.add_self_attention(H, d, S + 2, 1e-12, wq, wk, wv, bias, one, nil)
        got = net.forward_layers(0, 1, x, mask=mask, forward_only=False)
    y = (heads_output(x, wq, wk, wv, bias, mask) + x).real
    t = y - y.mean(-1, keepdims=True)
    want = t / np.sqrt((t * t).mean(-1, keepdims=True) + 1e-12)
    assert np.all(got.imag == 0)
    assert np.max(np.abs(got.real - want)) < 1e-12 * np.max(np.abs(want))


@pytest.mark.parametrize("B,S,H,dh,at", [(2, 100, 2, 16, 40), (1, 33, 1, 64, 32), (130, 40, 4, 20, 39), (1, 300, 2, 32, 299),
                                         (40, 200, 5, 24, 130), (1, 70, 2, 128, 66)])
def test_a_later_row_that_is_not_finite_reaches_the_earlier_ones(B, S, H, dh, at):
    """A masked key has weight 0, and 0 times a value that is not finite is
    NaN (utils/matrix.rs:356-380 sums over every key): the tiled kernel, which
    skips masked tiles, against the one-row-per-block form."""
    d = H * dh
    r = np.random.default_rng(at)
    c = lambda *s: r.standard_normal(s) + 1j * r.standard_normal(s)  # noqa: E731
    wq, wk, wv = (c(H, d, dh) / np.sqrt(2 * d) for _ in range(3))
    x = c(B, S, d)
    x[0, at, 3] = complex(np.inf, 0.5)
    mask = np.ones((B, S), np.uint32)
    mask[:, 0] = 0  # a padded row stays 0
    out = []
    for plan in (1, 0):
        with ra.Network(0) as net:
            net.add_self_attention(H, d, S, 1e-12, wq, wk, wv, 0.3 * np.ones((H, S, S)))
            net.set_decode_plan(plan)
            out.append(net.forward_layers(0, 1, x, mask=mask, forward_only=False))
    tiled, rows = out
    assert np.array_equal(np.isnan(tiled), np.isnan(rows))
    assert np.isnan(rows[0, 1:].real).all() and np.isfinite(rows[0, 0]).all() and np.isfinite(rows[1:]).all()
    live = np.isfinite(rows)
    assert np.max(np.abs(tiled[live] - rows[live])) < 1e-12 * np.max(np.abs(rows[live]))
