"""Layers of up to 512 units run chained in one launch, wider ones in a launch
each.  A narrow model and the same model with more units whose weights are 0
form the same sums in the same order (what is added is 0), so the two paths
agree bit for bit: outputs, loss, gradients and training.
"""
import numpy as np
import pytest

from bsim_amd import surrogate

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

WIDE = 576


def spans(hidden, layers, out_dim):
    """(rows, columns, weight offset, bias offset) of each layer, and the length."""
    dims = [64] + [hidden] * layers + [(out_dim + 63) // 64 * 64]
    s, off = [], 0
    for k, n in zip(dims, dims[1:]):
        s.append((n, k, off, off + n * k))
        off += n * k + n
    return s, off


def widen(p, narrow, wide, total):
    q = np.zeros(total, np.float32)
    for (n, k, w, b), (N, K, W, B) in zip(narrow, wide):
        q[W:W + N * K].reshape(N, K)[:n, :k] = p[w:w + n * k].reshape(n, k)
        q[B:B + n] = p[b:b + n]
    return q


@pytest.mark.parametrize("in_dim,hidden,layers,out_dim,batch", [
    (1, 64, 1, 1, 256), (8, 192, 2, 37, 256), (33, 256, 4, 257, 768), (64, 320, 3, 64, 512),
    (5, 448, 2, 130, 256), (8, 512, 4, 200, 1280), (17, 512, 9, 512, 256)])
def test_chained_equals_layered(in_dim, hidden, layers, out_dim, batch):
    say(f"[gpu] chained {in_dim}-{hidden}x{layers}-{out_dim} batch {batch}")
    rng = np.random.Generator(np.random.PCG64(hidden + layers))
    kw = dict(in_dim=in_dim, layers=layers, out_dim=out_dim, max_batch=batch)
    m, v = surrogate.MLP(hidden=hidden, **kw), surrogate.MLP(hidden=WIDE, **kw)
    narrow, _ = spans(hidden, layers, out_dim)
    wide, total = spans(WIDE, layers, out_dim)
    p = m.get_params()
    for n, k, w, b in narrow:                   # biases, so that few activations are 0 by themselves
        p[b:b + n] = rng.normal(0.0, 0.1, n)
    m.set_params(p)
    p = m.get_params()                          # with the padding cleared
    v.set_params(widen(p, narrow, wide, total))
    for rows in (0, 1, 31, 32, 33, batch, 2 * batch + 65, 4000):
        x = rng.normal(size=(rows, in_dim)).astype(np.float32)
        np.testing.assert_array_equal(m.predict(x), v.predict(x))
    x = rng.normal(size=(batch, in_dim)).astype(np.float32)
    y = rng.normal(size=(batch, out_dim)).astype(np.float32)
    (g, loss), (h, wloss) = m.gradients(x, y), v.gradients(x, y)
    assert loss == wloss and np.any(g != 0)
    np.testing.assert_array_equal(widen(g, narrow, wide, total), h)
    for z in (m, v):
        z.set_data(x, y)
    rows = rng.integers(0, batch, (3, batch)).astype(np.int32)
    np.testing.assert_array_equal(m.train(rows, batch, 1e-3), v.train(rows, batch, 1e-3))
    np.testing.assert_array_equal(widen(m.get_params(), narrow, wide, total), v.get_params())
    m.close()
    v.close()
