"""The tiled MFMA product (gemm_mfma.hip, more than 64 rows) at the edges of
its 64x64 tiles and 8-wide K steps, with and without a split of K, on complex
rows and on the real rows a Norm leaves, against numpy.

Bound: a product of K terms summed in any order is within (K + 4) eps of
sum |a| |b| per part (the four real products add two such sums).
"""
from __future__ import annotations

import numpy as np
import pytest

import rustcrates_amd as ra

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps

# rows, K, N: one row past a tile, remainders of a K step, one tile, a split
# of every tile (fewer than 256 tiles), whole tiles and split ones (over 256)
SHAPES = [(65, 8, 64), (65, 9, 63), (127, 7, 65), (64 * 3, 100, 130), (70, 1024, 64), (130, 777, 96),
          (519, 264, 2304), (257 * 64, 16, 64)]
# at most 64 rows: the row-tile products, straight-line (512 and 768 of K) and looped
SKINNY = [(9, 512, 64), (33, 768, 33), (64, 512, 1000), (17, 300, 48), (64, 1000, 20), (20, 257, 17)]


def linear_net(d, n, seed, w=None):
    r = np.random.default_rng(seed)
    if w is None:
        w = r.standard_normal((d, n)) + 1j * r.standard_normal((d, n))
    b = r.standard_normal(n) + 1j * r.standard_normal(n)
    net = ra.Network(0)
    net.add_norm(d, 1e-5)
    net.add_linear(d, n, w, b)
    return net, w, b


def close(got, a, w, b):
    want = a @ w + b
    bound = (w.shape[0] + 4) * EPS * (np.abs(a) @ np.abs(w) + np.abs(b))
    for g, v in ((got.real, want.real), (got.imag, want.imag)):
        over = np.abs(g - v) - bound
        assert np.all(over <= 0), float(over.max())


@pytest.mark.parametrize("rows,k,n", SHAPES + SKINNY)
def test_tiled_product_on_complex_and_real_rows(rows, k, n):
    net, w, b = linear_net(k, n, rows + k + n)
    r = np.random.default_rng(rows)
    x = r.standard_normal((1, rows, k)) + 1j * r.standard_normal((1, rows, k))
    with net:
        y = net.forward_layers(1, 2, x, forward_only=False, d_out=n)[0]
        h = net.forward_layers(0, 1, x, forward_only=False)[0]  # real rows
        z = net.forward_layers(0, 2, x, forward_only=False, d_out=n)[0]
    assert np.all(h.imag == 0)
    close(y, x[0], w, b)
    close(z, h, w, b)


@pytest.mark.parametrize("rows,k", [(70, 40), (20, 512), (20, 300)])
def test_real_rows_meet_infinities_and_nan_as_complex_ones_do(rows, k):
    """A product with zero imaginary parts left out must still give NaN where 0 * (infinity or NaN) would."""
    n = 80
    r = np.random.default_rng(3)
    w = r.standard_normal((k, n)) + 1j * r.standard_normal((k, n))
    w[3, 2] = complex(np.inf, 1.0)
    w[39, 64] = complex(1.0, -np.inf)
    w[8, 79] = complex(np.nan, 1.0)
    w[7, 70] = complex(0.5, np.nan)
    net, w, b = linear_net(k, n, 4, w)
    x = r.standard_normal((1, rows, k)) + 1j * r.standard_normal((1, rows, k))
    with net:
        h = net.forward_layers(0, 1, x, forward_only=False)[0]
        z = net.forward_layers(0, 2, x, forward_only=False, d_out=n)[0]
    with np.errstate(invalid="ignore"):
        re = h.real @ w.real - h.imag @ w.imag
        im = h.real @ w.imag + h.imag @ w.real
    for got, want in ((z.real, re), (z.imag, im)):
        assert np.array_equal(np.isnan(got), np.isnan(want))
        inf = np.isinf(want)
        assert inf.any() and np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf])


@pytest.mark.parametrize("rows,d,V", [(70, 512, 9600), (130, 200, 6400), (65, 512, 64)])
def test_greedy_ids_of_a_split_last_round(rows, d, V):
    """The vocabulary product of more than 64 sequences forms each row's id in
    its epilogue: with whole tiles and split ones in one launch (150 column
    tiles of 2 row tiles, 100 of 3), and with every tile split."""
    r = np.random.default_rng(V)
    table = r.standard_normal((rows + 3, d)) + 1j * r.standard_normal((rows + 3, d))
    w = r.standard_normal((d, V)) + 1j * r.standard_normal((d, V))
    b = r.standard_normal(V) + 1j * r.standard_normal(V)
    ids = np.arange(2, rows + 2, dtype=np.uint32)[:, None]
    with ra.Network(0) as net:
        net.add_embedding(rows + 3, d, table)
        net.add_linear(d, V, w, b)
        net.add_softmax(ra.PRODUCTION)
        got, lg = net.generate(ids, lens=np.ones(rows, np.uint32), n_new=1, want_logits=True)
    x = table[ids[:, 0]]
    bound = (d + 4) * EPS * (np.abs(x) @ np.abs(w) + np.abs(b))
    lg = np.asarray(lg).reshape(rows, V)
    assert np.all(np.abs(lg - (x @ w + b).real) <= bound)
    assert np.array_equal(np.asarray(got).reshape(rows), V - 1 - np.argmax(lg[:, ::-1], axis=1))  # the last of equal ones
