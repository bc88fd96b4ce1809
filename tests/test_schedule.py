"""The order of the units does not change results, whatever it is made from: units
ranked every cycle, every third, never, and the schedule changed in mid-run, in
networks of more units than run at a time (smaller ones are not ranked).  Bit for bit
against the oracle."""
import numpy as np
import pytest

import oracle
from bsim_amd import api, netspec

from test_gpu_parity import DT, say
from test_step_units import connect, lif, sources

pytestmark = pytest.mark.gpu

TILE = 192


def network(npop, dmax, steps):
    n, s = 9408, 300
    rng = np.random.Generator(np.random.PCG64(100 * npop + dmax))
    b = netspec.Builder()
    for p in range(npop):
        base = p * (s + n)
        sources(b, s, steps, rng, 0.3 if p % 4 == 1 else 0.02)
        lif(b, n, rng)
        connect(b, base + np.repeat(np.arange(s), 300), base + s + rng.integers(0, n, 300 * s), rng, dmax, 0.05)
    return b.build()


# units past 512 with delays past 24 steps keep their order within a class; 52 populations
# run, and are ranked, in workgroups of eight wavefronts
@pytest.mark.parametrize("npop,dmax,steps,schedules", [
    (7, 3, 150, [[1], [3], [0, 5, 1, 0, 4, 2]]),
    (11, 30, 150, [[1], [0, 1, 3, 0, 2, 1]]),
    (52, 2, 40, [[1], [0, 3, 1, 0]])])
def test_schedules_of_ranked_units(npop, dmax, steps, schedules):
    spec = network(npop, dmax, steps)
    units = -(-spec.n // TILE)
    assert units > {7: 256, 11: 512, 52: 2560}[npop]
    o = oracle.run(spec, DT, steps, mode="csr", tile=256, threads=8)
    assert o.events > 10_000 and len(o.raster_ids) > 0
    net = api.Network.from_spec(spec)
    for sched in schedules:
        say(f"[gpu] schedule {sched} of {units} units, delays up to {dmax}, n={spec.n} s={spec.s}")
        sim = api.Simulation(net, DT, tile=TILE, rec_steps=steps)
        left = steps
        for i, r in enumerate(sched):
            sim.set_schedule(r)
            # portions of odd and even lengths; the last has what is left, past a graph's 64 cycles
            k = left if i + 1 == len(sched) else 7 + i % 3
            sim.step(k)
            left -= k
        sim.finish()
        sim.sync()
        counts, ids, _ = sim.raster()
        st = sim.state()
        assert np.array_equal(counts, o.raster_count) and np.array_equal(ids, o.raster_ids), sched
        for k in ("v", "ie", "ii"):
            assert np.array_equal(st[k].view(np.uint32), getattr(o, "final_" + k).view(np.uint32)), (sched, k)
        assert sim.events() == o.events, sched
        sim.close()
