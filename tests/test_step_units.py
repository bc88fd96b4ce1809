"""The step kernel at the sizes where its passes, slots and units change:
whole tiles and tiles in parts, a target with more events in a pass than it has
slots, a sub-row longer than a pass, more source ranges than one batch holds,
blocks of rows without a synapse into the unit, units that change XCD, networks of one
unit and many cycles per launch.  Bit for bit against the oracle, as everything the step computes is.
"""
import numpy as np
import pytest

import oracle
from bsim_amd import api, netspec

from test_gpu_parity import DT, assert_same, run_gpu, say

pytestmark = pytest.mark.gpu

LIF = netspec.lif_row(0.0, 0.0, 0.0, 0.02, 0.02, 3e-4, 5e-3, 8e-3, 1.0, 0.0)


def sources(b, n, steps, rng, p=0.3):
    """n array sources that fire at random cycles."""
    return b.population(np.zeros((n, netspec.LIF_NPARAM)), kind=netspec.ARRAY,
                        spikes=[np.nonzero(rng.random(steps) < p)[0] for _ in range(n)])


def lif(b, n, rng):
    rows = np.tile(LIF, (n, 1))
    rows[:, 9] = rng.uniform(0.3, 1.4, n)
    return b.population(rows)


def connect(b, pre, post, rng, dmax, scale):
    """Creation order (pre, delay): mixed signs, integer delays."""
    k = rng.integers(1, dmax + 1, len(pre))
    order = np.lexsort((post, k, pre))
    pre, post, k = pre[order], post[order], k[order]
    w = np.where(rng.random(len(pre)) < 0.4, -1.0, 1.0) * rng.uniform(0.0, scale, len(pre))
    b.connect(pre, post, w.astype(np.float32), k.astype(np.float32) * np.float32(DT),
              (w < 0).astype(np.int8))


def net(kind, steps):
    rng = np.random.Generator(np.random.PCG64(sum(map(ord, kind))))
    b = netspec.Builder()
    if kind == "one_target":            # every event of a pass on one target, ranks far past its slots
        s = 2600
        sources(b, s, steps, rng, 0.5)
        lif(b, 3, rng)
        connect(b, np.repeat(np.arange(s), 2), np.full(2 * s, s + 1), rng, 2, 2e-3)
    elif kind == "long_rows":           # sub-rows of up to 2,300 events, longer than a pass
        s, n = 12, 1150
        sources(b, s, steps, rng)
        lif(b, n, rng)
        pre = np.repeat(np.arange(s), 2 * n)
        post = s + np.tile(np.repeat(np.arange(n), 2), s)
        k = np.ones(len(pre))
        w = rng.uniform(-0.02, 0.03, len(pre)).astype(np.float32)
        b.connect(pre, post, w, k.astype(np.float32) * np.float32(DT), (w < 0).astype(np.int8))
    elif kind == "many_ranges":         # 290 source ranges: three batches
        s, n, gap = 290, 150, 300
        sources(b, s * gap, 1, rng, 0.0)
        b.arr[:s * gap:gap] = [np.nonzero(rng.random(steps) < 0.4)[0].astype(np.int32) for _ in range(s)]
        lif(b, n, rng)
        connect(b, np.repeat(np.arange(s) * gap, 40), s * gap + rng.integers(0, n, 40 * s), rng, 4, 0.05)
    else:                               # "empty_blocks": 3,000 active rows, few with a synapse into a unit
        s, n = 3000, 700
        sources(b, s, steps, rng, 0.6)
        lif(b, n, rng)
        connect(b, np.arange(s), s + np.where(np.arange(s) < s - 40, n - 1, rng.integers(0, n, s)), rng, 1, 0.01)
    return b.build()


@pytest.mark.parametrize("tile", [192, 384, 768, 1536])
@pytest.mark.parametrize("kind", ["one_target", "long_rows", "many_ranges", "empty_blocks"])
def test_edges_of_passes_and_slots(kind, tile):
    steps = 40
    spec = net(kind, steps)
    rec = [spec.n - 3, spec.n - 2, spec.n - 1]
    say(f"[gpu] {kind} n={spec.n} s={spec.s} tile={tile}")
    r = run_gpu(spec, steps, rec, tile)
    o = oracle.run(spec, DT, steps, rec_ids=rec, mode="csr", tile=256, threads=8)
    assert o.events > 1000
    assert_same(r, o, kind)


@pytest.mark.parametrize("npop,tile", [(2, 192), (7, 384)])
def test_whole_tiles(npop, tile):
    """Enough tiles that each is one unit, and the tile after the last population ragged."""
    spec = netspec.standard(npop=npop, n=10007, fanout=24, w0=12.0, dmax=7, drive_rate_hz=200.0,
                            n_drive=500, drive_fanout=40, drive_w=2.0, seed=5, i_offset=(14.5, 16.5))
    steps, rec = 220, [600, spec.n - 1]
    say(f"[gpu] whole tiles npop={npop} n={spec.n} s={spec.s} tile={tile}")
    r = run_gpu(spec, steps, rec, tile)
    o = oracle.run(spec, DT, steps, rec_ids=rec, mode="csr", tile=256, threads=8)
    assert o.events > 10_000
    assert_same(r, o, "whole tiles")


@pytest.mark.parametrize("npop,active", [(11, 1), (11, 11), (52, 9)])
def test_ranked_units(npop, active):
    """More units than run at a time, ranked every other cycle: populations of
    which one, some or every one is active; with 52 also in workgroups of eight
    wavefronts."""
    n, s, steps = 9408, 300, 40
    rng = np.random.Generator(np.random.PCG64(active))
    b = netspec.Builder()
    for p in range(npop):
        base = p * (s + n)
        sources(b, s, steps, rng, 0.3 if p < active else 0.01)
        lif(b, n, rng)
        connect(b, base + np.repeat(np.arange(s), 400), base + s + rng.integers(0, n, 400 * s), rng, 2, 0.05)
    spec = b.build()
    rec = [s, s + n - 1, spec.n - 1]
    say(f"[gpu] ranked units npop={npop} active={active} n={spec.n} s={spec.s}")
    r = run_gpu(spec, steps, rec, 192)
    o = oracle.run(spec, DT, steps, rec_ids=rec, mode="csr", tile=256, threads=8)
    assert o.events > 10_000
    assert_same(r, o, "ranked units")


@pytest.mark.parametrize("tile,dmax,n", [(192, 3, 1), (192, 3, 64), (192, 3, 65), (192, 7, 192), (192, 2, 193),
                                         (384, 12, 128), (384, 12, 129), (768, 40, 256), (768, 63, 257)])
def test_one_unit(tile, dmax, n):
    """Networks of one unit take up to 64 cycles per launch, in the last case of
    each pair one more neuron makes two."""
    steps, s = 150, max(n // 4, 1) if n > 1 else 0
    rng = np.random.Generator(np.random.PCG64(n))
    b = netspec.Builder()
    if s:
        sources(b, s, steps, rng)
    lif(b, n - s, rng)
    if s:
        connect(b, rng.integers(0, n, 12 * n), s + rng.integers(0, n - s, 12 * n), rng, dmax, 0.2)
    else:
        connect(b, np.zeros(3, int), np.zeros(3, int), rng, dmax, 0.2)
    spec = b.build()
    rec = sorted({0, n // 2, n - 1})
    say(f"[gpu] one unit tile={tile} n={n}")
    r = run_gpu(spec, steps, rec, tile)
    assert_same(r, oracle.run(spec, DT, steps, rec_ids=rec, mode="csr", tile=256, threads=8), "one unit")
    sim = api.Simulation(api.Network.from_spec(spec), DT, tile=tile)
    for k in (1, 2, 64, 1, 65, 17):             # cycles in other portions
        sim.step(k)
    sim.finish()
    sim.sync()
    st = sim.state()
    for k in ("v", "ie", "ii", "refrac"):
        assert np.array_equal(st[k], r[k]), k
    assert sim.events() == r["events"]
    sim.close()


@pytest.mark.parametrize("npop", [26, 28])
def test_deep_delays_of_many_units(npop):
    """Delays past 24 steps with more than 341 tiles of 768 are laid out in tiles
    of twice the size (28 populations); what the caller sees stays."""
    n, s, steps, dmax, tile = 9600, 200, 60, 30, 768
    rng = np.random.Generator(np.random.PCG64(npop))
    b = netspec.Builder()
    for p in range(npop):
        base = p * (s + n)
        sources(b, s, steps, rng, 0.1 if p % 3 else 0.4)
        lif(b, n, rng)
        connect(b, base + np.repeat(np.arange(s), 300), base + s + rng.integers(0, n, 300 * s), rng, dmax, 0.1)
    spec = b.build()
    rec = [s, s + n - 1, spec.n - 1]
    say(f"[gpu] deep delays npop={npop} n={spec.n} s={spec.s}")
    r = run_gpu(spec, steps, rec, tile)
    assert r["info"]["tile"] == tile and r["info"]["ntiles"] == -(-spec.n // tile)
    o = oracle.run(spec, DT, steps, rec_ids=rec, mode="csr", tile=256, threads=8)
    assert o.events > 10_000
    assert_same(r, o, "deep delays")
