"""FP32 steps bit for bit: the order of a vertex's sums and every rounding of its
solve are part of the result, since a contact leaves static friction at the last
bit and its vertex then moves by millimetres.  The recorded values are those of
the FP32 kernels as the framework first had them (one launch per colour phase;
deformation gradient and cofactors per incidence, quotients in the 3x3 and 6x6
solves, lane sums as a butterfly from L / 2 down to 1, a vertex's or body's
dynamic contacts added one after the other behind its other terms); every other
path (the resident solve, batches) has to reproduce them."""
from pathlib import Path

import numpy as np
import pytest

from avbd_amd import _lib, scenes

pytestmark = pytest.mark.gpu

GOLDEN = Path(__file__).resolve().parent / "golden" / "fp32_steps.npz"
# name: (cells per edge from, to, cubes, damping), lanes per vertex
CASES = {f"{kind}_{lanes}": (*size, lanes)
         for lanes in (4, 8, 16, 32) for kind, size in (("batch", (1, 4, 6, 0.0)), ("damped", (3, 3, 1, 1e-3)))}
CONTACTS = {f"{name}_{lanes}": (name, lanes) for name, lanes in
            (("hail", 8), ("hail", 32), ("ball", 16), ("stack", 4), ("stack", 8), ("stack", 32), ("pile", 8))}
STEPS, ITERS = 25, 10


def scene_of(n_min, n_max, cubes, kd):
    sc = scenes.cube_batch(n_scenes=cubes, n_min=n_min, n_max=n_max)
    for k, m in enumerate(sc.meshes):
        m.rest[:, 1] += 0.002 * (k + 1) - m.rest[:, 1].min()
        m.v0 = np.tile([0.3, -1.0, 0.1 * k], (len(m.rest), 1))   # slides: contacts stick and slip
        m.kd = kd
    sc.iters = ITERS
    return sc


def contact_scene(name):
    sc = {"hail": lambda: scenes.hail_on_block(n=6, grid=3), "ball": scenes.ball_on_block, "stack": scenes.block_stack,
          "pile": scenes.sphere_pile}[name]()
    for k, sphere in enumerate(sc.spheres):   # roll and slide
        sphere.v0 = (0.2, -0.4, 0.05 * k)
    return sc


def run(case, **kw):
    from avbd_amd.sim import Simulation
    *size, lanes = CASES.get(case) or CONTACTS[case]
    sc = scene_of(*size) if case in CASES else contact_scene(*size)
    sim = Simulation(sc, lanes_per_vertex=lanes, block_size=128, **kw)
    sim.setup()
    sim.update(STEPS)
    x, v = sim.ctx.state()
    return x.astype(np.float32), v.astype(np.float32)


@pytest.mark.parametrize("flags", [0, _lib.FLAG_NO_PERSISTENT])
@pytest.mark.parametrize("case", sorted(CASES) + sorted(CONTACTS))
def test_fp32_steps_are_bit_for_bit_the_recorded_ones(case, flags):
    print(f"[gpu-test] rounding {case} flags {flags}", flush=True)
    x, v = run(case, flags=flags)
    with np.load(GOLDEN) as g:
        assert np.array_equal(x, g[case + "_x"])
        assert np.array_equal(v, g[case + "_v"])
