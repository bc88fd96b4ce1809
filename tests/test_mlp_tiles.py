"""Products and weight gradients of wide layers run in bands of tiles, and where a
layer's operands are very large in tiles of 128 x 128.  A wide model made of copies
of a narrow one, copy r with activations 2^s_r times as large, has outputs and
gradients that are the narrow model's times powers of two, block by block, bit for
bit: what is added otherwise is 0, and scaling by a power of two rounds nothing.
"""
import numpy as np
import pytest

from bsim_amd import surrogate

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

H = 64          # units and outputs of the narrow model
DIN = 8


def split(p, hidden, out):
    """[(W, b)] of the layers as views of the flat parameters."""
    dims, r, off = [64, hidden, hidden, out], [], 0
    for k, n in zip(dims, dims[1:]):
        r.append((p[off:off + n * k].reshape(n, k), p[off + n * k:off + n * k + n]))
        off += n * k + n
    assert off == len(p)
    return r


# tiles of 64 x 64 in bands whose last is short; of 128 x 128, even and with a short band
@pytest.mark.parametrize("copies,outs,batch", [(17, 16, 1280), (32, 32, 24576), (34, 32, 24576)])
def test_copies_of_a_narrow_model(copies, outs, batch):
    say(f"[gpu] copies {copies} x {H} units, {outs} x {H} outputs, batch {batch}")
    rng = np.random.Generator(np.random.PCG64(copies))
    kw = dict(in_dim=DIN, layers=2, max_batch=batch)
    m = surrogate.MLP(hidden=H, out_dim=H, **kw)
    v = surrogate.MLP(hidden=copies * H, out_dim=outs * H, **kw)
    p, q = m.get_params(), np.zeros_like(v.get_params())
    for w, b in split(p, H, H):
        b[:] = rng.normal(0.0, 0.1, len(b))
    m.set_params(p)
    narrow, wide = split(p, H, H), split(q, copies * H, outs * H)
    scale = 2.0 ** (np.arange(copies) * 3 % 8)
    for c in range(copies):
        x = slice(c * H, c * H + H)
        s = np.float32(scale[c])
        wide[0][0][x], wide[0][1][x] = narrow[0][0] * s, narrow[0][1] * s
        wide[1][0][x, x], wide[1][1][x] = narrow[1][0], narrow[1][1] * s
        if c < outs:
            wide[2][0][x, x], wide[2][1][x] = narrow[2][0] / s, narrow[2][1]
    v.set_params(q)
    x = rng.normal(size=(batch, DIN)).astype(np.float32)
    y = rng.normal(size=(batch, H)).astype(np.float32)
    for rows in (1, 300):
        np.testing.assert_array_equal(v.predict(x[:rows]), np.tile(m.predict(x[:rows]), outs))
    ywide = np.tile(y, outs)
    g, loss = m.gradients(x, y)
    h, wloss = v.gradients(x, ywide)
    assert np.any(g != 0) and abs(loss - wloss) <= 3e-5 * loss     # sums of some 220 roundings each
    # d loss / d outputs has 1 / outs; unit copy i's gradient 2^-s_i, its inputs from copy j 2^s_j
    gn, gw = split(g, H, H), split(h, copies * H, outs * H)
    for l in range(3):
        to = np.where(np.arange(copies) < outs, 1.0 / scale, 0.0) if l < 2 else np.ones(outs)
        of = scale if l > 0 else np.ones(1)
        f = (np.outer(to, of) / outs).astype(np.float32)
        n, k = gn[l][0].shape
        blocks = gw[l][0].reshape(len(to), n, len(of), k)
        np.testing.assert_array_equal(blocks, f[:, None, :, None] * gn[l][0][None, :, None, :])
        np.testing.assert_array_equal(gw[l][1].reshape(len(to), n),
                                      (to / outs).astype(np.float32)[:, None] * gn[l][1])

    # Adam's first step from these gradients; every rounding of the step is 2^-24 of it
    # or of the parameter, and there are about ten
    v.set_data(x, ywide)
    lr = 1e-3
    v.train(np.arange(batch, dtype=np.int32)[None], batch, lr)
    after = v.get_params()
    b1, b2, eps = (float(np.float32(z)) for z in (v.cfg.beta1, v.cfg.beta2, v.cfg.eps))
    h64 = h.astype(np.float64)
    mh, vh = (1 - b1) * h64 / (1 - b1), (1 - b2) * h64 * h64 / (1 - b2)
    want = q - np.float32(lr) * (mh / (np.sqrt(vh) + eps))
    assert np.all(np.abs(after - want) <= 1e-6 * lr + 2.0 ** -23 * np.abs(want))
    # the bf16 copies that the step left are those of its parameters
    u = surrogate.MLP(hidden=copies * H, out_dim=outs * H, **kw)
    u.set_params(after)
    np.testing.assert_array_equal(u.predict(x[:300]), v.predict(x[:300]))
    np.testing.assert_array_equal(u.gradients(x, ywide)[0], v.gradients(x, ywide)[0])
    for z in (m, v, u):
        z.close()
