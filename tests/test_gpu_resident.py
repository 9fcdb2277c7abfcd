"""The resident solve (every iteration of a stretch in one launch, the patches
of a scene in the LDS of workgroups that exchange boundary positions) equals
one launch per phase bit for bit at the same lanes per vertex, whatever the
partition: scenes of one patch and of many, patches of odd sizes, particles
without a free neighbour, damping, ground contacts, batches of scenes of
different sizes, odd iteration counts, and launches that alternate between the
exchange and the path for a device that cannot hold a scene's patches at once."""
import numpy as np
import pytest

from avbd_amd import _lib, scenes

pytestmark = pytest.mark.gpu


def scene_of(kind, n):
    if kind == "hang":
        sc = scenes.hanging_cube(n=n)
    elif kind == "damped":
        sc = scenes.dropped_cube(n=n, height=0.01)
        for m in sc.meshes:
            m.kd = 1e-3
    elif kind in ("batch", "crowd"):
        sc = scenes.cube_batch(n_scenes=n, n_min=1, n_max=9 if kind == "batch" else 14)
        for m in sc.meshes:
            m.rest[:, 1] += 0.01 - m.rest[:, 1].min()
    else:
        sc = scenes.dropped_cube(n=n, height=0.01)
    return sc


# a single cell, a cube below one patch, just above it, tens of patches, ragged
# ones; lanes below and above the number of 32-bit pieces of a position; patches that fill
# the LDS and have more items in a phase than 512 threads hold groups (FP32: 1,024 threads,
# FP64: a group takes a second item), one scene and many, damped and not; a crowd's
# larger cubes do not fit as they are first cut
CASES = [("hang", 1, 8), ("hang", 2, 4), ("drop", 5, 16), ("drop", 6, 32), ("drop", 13, 8), ("damped", 3, 8),
         ("damped", 9, 32), ("batch", 7, 8), ("batch", 40, 4), ("drop", 32, 16), ("drop", 32, 32), ("damped", 28, 32),
         ("crowd", 400, 8), ("crowd", 400, 32)]


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("kind,n,lanes", CASES)
def test_resident_equals_one_launch_per_phase(kind, n, lanes, fp64):
    from avbd_amd.sim import Simulation
    print(f"[gpu-test] resident {kind} {n} lanes {lanes} fp64 {fp64}", flush=True)
    sc = scene_of(kind, n)
    sc.iters = 7
    kw = dict(fp64_state=fp64, lanes_per_vertex=lanes, block_size=128)
    runs = [Simulation(sc, flags=f, **kw)
            for f in (_lib.FLAG_NO_PERSISTENT, 0, _lib.FLAG_RESIDENT_ALONE, _lib.FLAG_NO_GRAPH)]
    for r in runs:
        r.setup()
        assert (r.ctx.persistent_grid() > 0) == (r is not runs[0])
    for k in range(3):
        for r in runs:
            r.update(3)
        x0, v0 = runs[0].ctx.state()
        assert np.isfinite(x0).all()
        for j, r in enumerate(runs[1:]):
            x, v = r.ctx.state()
            assert np.array_equal(x, x0) and np.array_equal(v, v0), (k, j)
    if kind != "hang":
        ref = bytes(runs[0].ctx.ground_records())
        assert all(bytes(r.ctx.ground_records()) == ref for r in runs[1:])


@pytest.mark.parametrize("kind,n,check", [("drop", 6, 1), ("drop", 7, 5), ("drop", 13, 10), ("batch", 9, 3),
                                          ("batch", 30, 150)])
def test_resident_stops_where_one_launch_per_phase_stops(kind, n, check):
    """Residual target: the same iteration counts and positions, with scenes of
    a batch that stop at different checks and steps at the budget (203 is no
    multiple of a launch's intervals).  The residual sums differ in order only
    (at most 4000 FP64 terms >= 0 per scene: 1e-12)."""
    from avbd_amd.sim import Simulation
    print(f"[gpu-test] resident residual {kind} {n} every {check}", flush=True)
    sc = scene_of(kind, n)
    kw = dict(fp64_state=True, lanes_per_vertex=8, block_size=128, residual_target=(1e-4, 203, check))
    runs = [Simulation(sc, flags=f, **kw) for f in (_lib.FLAG_NO_PERSISTENT, 0, _lib.FLAG_RESIDENT_ALONE)]
    for r in runs:
        r.setup()
        r.update(4)
    s0, h0 = runs[0].ctx.stats(), runs[0].ctx.residual_history()
    for r in runs[1:]:
        s = r.ctx.stats()
        assert (s.iterations_total, s.last_step_iterations) == (s0.iterations_total, s0.last_step_iterations)
        assert np.allclose(r.ctx.residual_history(), h0, rtol=1e-12, atol=0)
        assert np.allclose(r.ctx.residual_history(worst_scene=True), runs[0].ctx.residual_history(worst_scene=True),
                           rtol=1e-12, atol=0)
        assert (s.steps_at_budget, s.vertex_updates) == (s0.steps_at_budget, s0.vertex_updates)
        assert np.array_equal(r.ctx.scene_iterations(), runs[0].ctx.scene_iterations())
        assert np.array_equal(r.positions(), runs[0].positions())


# one element; bundles of several short rods with a remainder; components of
# more particles than a bundle's share; a phase of more pairs than one
# workgroup holds (there is then one launch per phase)
@pytest.mark.parametrize("nx,nz,segments,jointed", [(1, 1, 1, False), (3, 3, 2, True), (5, 7, 9, False), (2, 2, 200, True),
                                                    (1, 1, 600, False)])
def test_bundles_of_rods_match_one_launch_per_phase(nx, nz, segments, jointed, oracle):
    """Oriented particles: the bundles' solve adds the two elements of a node in
    two lanes, so it differs from one launch per phase by the rounding of
    that sum; against the float64 oracle neither may be much further off than the
    other (twice, plus 1e-6 of the size: a few roundings of a position of 1)."""
    from avbd_amd.sim import Simulation
    print(f"[gpu-test] bundles {nx}x{nz} rods of {segments} jointed {jointed}", flush=True)
    sc = scenes.rod_grid(nx, nz, segments, iters=5, tip_joint=jointed)
    o = oracle.from_scene(sc)
    o.step(3)
    xo, err = o.positions(), []
    for kw in (dict(flags=_lib.FLAG_NO_PERSISTENT), dict(), dict(use_graph=False)):
        s = Simulation(sc, **kw)
        s.setup()
        s.update(3)
        err.append(np.abs(s.positions() - xo).max())
    print(f"[gpu-test]   off the oracle: per phase {err[0]:.2e}, bundles {err[1]:.2e}", flush=True)
    assert err[1] <= 2 * err[0] + 1e-6
    assert err[1] == err[2]


def test_scenes_that_wait_for_a_part_of_the_device_are_not_given_up():
    """Three scenes whose patches fill 1.4 times the device, many iterations per
    step: part of the third starts at once and waits for the first two.  A wait
    as long as their 6,000 iterations (90 ms) made it give up and run on one
    workgroup (18 s); the stretch is cut into launches instead.  At most three
    times what one launch per phase takes."""
    import time
    from avbd_amd.sim import Simulation
    print("[gpu-test] three scenes, 6,000 iterations", flush=True)
    sc = scenes.cube_batch(n_scenes=3, n_min=20, n_max=20)
    sc.iters = 6000
    took, x = [], []
    for f in (0, _lib.FLAG_NO_PERSISTENT):
        s = Simulation(sc, fp64_state=True, flags=f, lanes_per_vertex=8, block_size=128)
        s.setup()
        s.update(1)
        s.ctx.synchronize()
        t = time.perf_counter()
        s.update(1)
        x.append(s.positions())
        took.append(time.perf_counter() - t)
    print(f"[gpu-test]   resident {took[0] * 1e3:.0f} ms, per phase {took[1] * 1e3:.0f} ms", flush=True)
    assert np.array_equal(x[0], x[1])
    assert took[0] <= 3 * took[1]
