"""The step kernel's workgroups of eight wavefronts, which networks of 2,560 units and
more use, at the sizes where its passes, slots and batches change: the networks of
test_step_units with idle neurons up to that many units, and sweeps of tiny networks
each padded to whole tiles, in units of 64 and 128 targets.  Bit for bit against the
oracle."""
import numpy as np
import pytest

import oracle
from bsim_amd import api, netspec, sweep

from test_gpu_parity import DT, assert_same, run_gpu, say
from test_step_units import net

pytestmark = pytest.mark.gpu

UNITS = 2560


@pytest.mark.parametrize("kind", ["one_target", "long_rows", "many_ranges", "empty_blocks"])
def test_edges_of_passes_and_slots(kind):
    steps, tile = 40, 192
    spec = net(kind, steps)
    n = spec.n
    idle = (UNITS + 1) * tile - 5 - n           # array sources that never fire
    spec.kind = np.concatenate([spec.kind, np.full(idle, netspec.ARRAY, spec.kind.dtype)])
    spec.lif = np.concatenate([spec.lif, np.zeros((idle, spec.lif.shape[1]), spec.lif.dtype)])
    spec.arr_off = np.concatenate([spec.arr_off, np.full(idle, spec.arr_off[-1], spec.arr_off.dtype)])
    if spec.bern_p is not None:
        spec.bern_p = np.concatenate([spec.bern_p, np.zeros(idle, spec.bern_p.dtype)])
    rec = [n - 3, n - 2, n - 1, spec.n - 1]
    say(f"[gpu] eight wavefronts: {kind} n={spec.n} s={spec.s}")
    r = run_gpu(spec, steps, rec, tile)
    assert -(-spec.n // tile) >= UNITS
    o = oracle.run(spec, DT, steps, rec_ids=rec, mode="csr", tile=256, threads=8)
    assert o.events > 1000
    assert_same(r, o, kind)


@pytest.mark.parametrize("tile", [192, 384])
def test_padded_sweep(tile):
    """860 networks laid out one by one: each fills a tile of three units."""
    count, steps = 860, 120
    rng = np.random.Generator(np.random.PCG64(tile))
    pts = []
    for i in range(count):
        k = 60 if i % 43 == 7 else 3
        sizes = [int(x) for x in rng.integers(k, k + 4, 2)]
        pts.append(sweep.Point(sizes=sizes, fan_in=k, w0=1.5, inh_frac=0.2, dmax=int(rng.integers(2, 12)),
                               drive_rate_hz=400.0, n_drive=k, drive_fan_in=k, drive_w=2.0, seed=1000 + i))
    n = sum(p.n for p in pts)
    assert 3 * -(-n // tile) <= 256 * (tile // 192) and max(p.n for p in pts) <= 192
    say(f"[gpu] eight wavefronts: {count} networks of {n} neurons in units of {tile // 3}")
    sim, first = api.Simulation.from_chains([p.kwargs() for p in pts], DT, tile=tile, rec_steps=steps,
                                            part_synapses=1)
    assert sim.n == count * tile
    sim.step(steps)
    sim.finish()
    sim.sync()
    counts, ids, _ = sim.raster()
    st, events = sim.state(), sim.events()
    sim.close()
    assert events > 10_000
    got = sweep.split_raster(counts, ids, first, np.array([p.n for p in pts]))
    total = 0
    for k, p in enumerate(pts):             # each against the oracle, alone: an exported network has one seed
        alone = api.Network()
        alone.add_chain(**p.kwargs())
        o = oracle.run(alone.export_spec(), DT, steps, mode="csr", tile=256, threads=1)
        total += o.events
        for c, want in enumerate(o.raster()):
            np.testing.assert_array_equal(got[k][c], want, err_msg=f"network {k} cycle {c}")
        z = slice(first[k], first[k] + p.n)
        for x in ("v", "ie", "ii"):
            assert np.array_equal(st[x][z].view(np.uint32), getattr(o, "final_" + x).view(np.uint32)), (k, x)
    assert total == events
