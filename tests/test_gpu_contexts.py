"""Several contexts stepped at once, each on its own thread and stream."""
import threading
import time

import numpy as np
import pytest

from avbd_amd import scenes

pytestmark = pytest.mark.gpu


def build(n, target, **kw):
    from avbd_amd.sim import Simulation
    s = Simulation(scenes.dropped_cube(n=n, height=0.02), lanes_per_vertex=8, block_size=128, residual_target=target, **kw)
    s.setup()
    s.update(2)
    s.positions()
    return s


def wall(sims, steps):
    """Seconds of `steps` steps of every context, all at once."""
    def go(s):
        for _ in range(steps):
            s.update(1)
        s.positions()
    threads = [threading.Thread(target=go, args=(s,)) for s in sims]
    t = time.perf_counter()
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    return time.perf_counter() - t


# contexts of which one fills the device (one patch per CU), many small ones that fit side by
# side, and a mix; to a residual and at a fixed count, by graphs and eagerly
@pytest.mark.parametrize("cells,fp64,target,graph", [
    ((16, 20, 24), True, (1e-4, 300, 10), True), ((20,) * 6, True, (1e-4, 300, 10), True),
    ((28,) * 3, True, (1e-4, 300, 10), True), ((20,) * 4, True, None, True), ((32, 32), False, None, True),
    ((8,) * 6, True, (1e-4, 100, 10), True), ((24, 6, 13), False, None, False)])
def test_contexts_on_threads_step_as_they_do_alone(cells, fp64, target, graph):
    """The patches of a scene wait for each other, so contexts that do not fit the
    device together take turns; none may end up waiting for another's: a cluster
    that gives up after its 50 ms runs on one workgroup, and without the turns half
    of the runs of the first three took four to six times as long as one context
    after the other.  The same results as alone, in at most three times that time,
    plus 20 ms for the host."""
    print(f"[gpu-test] contexts {cells} fp64 {fp64} target {target} graph {graph}", flush=True)
    steps = 12 if target else 60
    alone, apart = [], 0.0
    for n in cells:
        s = build(n, target, fp64_state=fp64, use_graph=graph)
        apart += wall([s], steps)
        alone.append((s.positions(), s.ctx.stats().iterations_total))
        s.ctx.close()
    sims = [build(n, target, fp64_state=fp64, use_graph=graph) for n in cells]
    together = wall(sims, steps)
    print(f"[gpu-test]   one after the other {apart * 1e3:.1f} ms, at once {together * 1e3:.1f} ms", flush=True)
    for s, (x, its) in zip(sims, alone):
        assert np.array_equal(s.positions(), x)
        assert s.ctx.stats().iterations_total == its
    assert together <= 3 * apart + 0.02
