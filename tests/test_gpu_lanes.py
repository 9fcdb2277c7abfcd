"""Lanes per vertex that the caller does not give: every path of a context sums a
vertex in the same order, so what runs a step (resident or per phase, timed or
not, quiet or with contacts in play) does not show in its result, and the
reported lanes reproduce it."""
import numpy as np
import pytest

from avbd_amd import _lib, scenes

pytestmark = pytest.mark.gpu


def two_cubes():
    """Two cubes that start apart and meet face to face."""
    sc = scenes.Scene("two_cubes", iters=10, rho=0.95, g=0.0, contact_margin=1e-3, self_collision=True, batch=False)
    for side in (-1.0, 1.0):
        rest, tets = scenes.kuhn_cube(3)
        x = 0.3 * rest + np.array([0.5, 0.0 if side < 0 else 0.32, 0.0])
        v = np.zeros_like(x)
        v[:, 1] = -0.3 * side
        sc.meshes.append(scenes.TetMesh(rest=x, tets=tets, triangles=scenes.surface_triangles(3), E=1e5, nu=0.3,
                                        density=1000.0, v0=v))
    return sc


# lanes the context ends with: below and above the line of each precision, damped on both sides of its first
@pytest.mark.parametrize("n,fp64,kd,lanes", [(5, False, 0.0, 32), (13, False, 0.0, 32), (24, False, 0.0, 8),
                                             (13, True, 0.0, 32), (16, True, 0.0, 8), (9, False, 1e-3, 32),
                                             (27, False, 1e-3, 16)])
def test_reported_lanes_reproduce_every_path(n, fp64, kd, lanes):
    from avbd_amd.sim import Simulation
    print(f"[gpu-test] lanes n {n} fp64 {fp64} kd {kd}", flush=True)
    sc = scenes.dropped_cube(n=n, height=0.004)
    sc.meshes[0].kd = kd
    sims = [Simulation(sc, fp64_state=fp64), Simulation(sc, fp64_state=fp64),
            Simulation(sc, fp64_state=fp64, flags=_lib.FLAG_NO_PERSISTENT)]
    for s in sims:
        s.setup()
        assert s.ctx.launch_config()[0] == lanes
    sims.append(Simulation(sc, fp64_state=fp64, lanes_per_vertex=lanes, block_size=128))
    sims[3].setup()
    sims[1].ctx.set_timing(True)
    for s in sims:
        s.update(4)
    x, v = sims[0].ctx.state()
    for s in sims[1:]:
        y, w = s.ctx.state()
        assert np.array_equal(x, y) and np.array_equal(v, w)


@pytest.mark.parametrize("fp64", [False, True])
def test_quiet_and_touching_steps_equal_one_launch_per_phase(fp64):
    """Dynamic contacts: resident steps while nothing touches, per phase after
    that, and resident again from a checkpoint of the quiet state."""
    from avbd_amd.sim import Simulation
    print(f"[gpu-test] quiet and touching steps, fp64 {fp64}", flush=True)
    sims = [Simulation(two_cubes(), fp64_state=fp64, flags=f) for f in (0, _lib.FLAG_NO_PERSISTENT)]
    saved, seen, touched = [], [], []
    for s in sims:
        s.setup()
        s.update(1)
        saved.append(s.ctx.save_checkpoint())
    for again in (False, True):
        for k in range(12):
            for s in sims:
                s.update(1)
            touched.append(len(sims[0].ctx.contacts(3)))
            (x, v), (y, w) = (s.ctx.state() for s in sims)
            assert np.array_equal(x, y) and np.array_equal(v, w), k
            if not again:
                seen.append((x, v))
            else:
                assert np.array_equal(x, seen[k][0]) and np.array_equal(v, seen[k][1]), k
        for s, c in zip(sims, saved):
            s.ctx.load_checkpoint(c)
    print(f"[gpu-test]   contacts per step {touched}", flush=True)
    assert touched[0] == 0 and touched[11] > 0


def test_step_mode_names_the_path_of_the_next_step():
    from avbd_amd.sim import Simulation
    print("[gpu-test] step mode", flush=True)
    cube, rods = scenes.dropped_cube(n=9, height=0.004), scenes.rod_grid(2, 2, 8, iters=5)
    grid = {}
    for name, sc, kw in (("cube", cube, {}), ("cube64", cube, dict(fp64_state=True)), ("rods", rods, {}),
                         ("target", cube, dict(residual_target=(1e-3, 100, 10))),
                         ("phases", cube, dict(flags=_lib.FLAG_NO_PERSISTENT)),
                         ("rod phases", rods, dict(flags=_lib.FLAG_NO_PERSISTENT)),
                         ("separate", cube, dict(separate_chebyshev=True)),
                         ("rods separate", rods, dict(separate_chebyshev=True)),
                         ("contacts", two_cubes(), {}), ("mixed", scenes.rod_on_block(), {})):
        s = Simulation(sc, **kw)
        s.setup()
        grid[name] = s.ctx.persistent_grid()
        s.ctx.set_timing(True)
        assert s.ctx.persistent_grid() == (grid[name] if name == "target" else 0)
        s.ctx.set_timing(False)
        if name == "contacts":
            s.update(1)
            grid["quiet"] = s.ctx.persistent_grid()
            s.update(12)
            grid["touching"] = s.ctx.persistent_grid()
        s.ctx.close()
    print(f"[gpu-test]   {grid}", flush=True)
    # 9^3 cells: (24 * 729 incidences + 8 * 1000 particles) / 1000 = 26 patches
    assert grid["cube"] == grid["cube64"] == grid["target"] == 26
    assert 0 < grid["rods"] <= 4
    assert grid["quiet"] > 0
    assert all(grid[k] == 0 for k in ("phases", "rod phases", "separate", "rods separate", "touching", "mixed"))
