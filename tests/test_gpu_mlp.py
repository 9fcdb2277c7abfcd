"""GPU tests of the learned warm start: the BF16 MFMA GEMM (lane layout and
transpositions against numpy), the network's forward and backward pass
against a numpy restatement fed the same bf16-rounded operands, training that
lowers the loss, and the warm-started solver against the plain one.

Tolerances: GEMM results equal an FP64 product of the bf16 inputs to FP32
accumulation error (rel 1e-5 of the row norm); gradients agree with the
numpy restatement to 2 % of each layer's gradient norm (bf16 rounding of the
back-propagated activations can flip at rounding boundaries)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def banner(msg):
    print(f"[gpu-test] {msg}", flush=True)


def bf16(a):
    """Round to bfloat16 (nearest even), returned as float32."""
    a = np.ascontiguousarray(a, dtype=np.float32)
    u = a.view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16
    return u.astype(np.uint32).view(np.float32)


def silu(z):
    return z / (1.0 + np.exp(-z))


def dsilu(z):
    s = 1.0 / (1.0 + np.exp(-z))
    return s * (1.0 + z * (1.0 - s))


IN, INP, HID, OUT, OUTP = 24, 32, 128, 3, 16
SHAPES = [(HID, INP), (HID, HID), (HID, HID), (OUTP, HID)]


def unpack(p):
    layers, off = [], 0
    for (o, i) in SHAPES:
        W = p[off:off + o * i].reshape(o, i)
        off += o * i
        b = p[off:off + o]
        off += o
        layers.append((W, b))
    norm = p[off:off + 2 * IN + 2 * OUT]
    return layers, norm


def reference_grads(p, X, T):
    """numpy restatement of the device forward/backward: bf16 operands,
    FP64 accumulation, MSE on the 3 outputs."""
    layers, norm = unpack(p)
    fm, fs, tm, ts = norm[:IN], norm[IN:2 * IN], norm[2 * IN:2 * IN + OUT], norm[2 * IN + OUT:]
    rows = X.shape[0]
    x = np.zeros((rows, INP), np.float32)
    x[:, :IN] = bf16((X - fm) / fs)
    t = (T - tm) / ts
    acts, zs = [x.astype(np.float64)], []
    h = x.astype(np.float64)
    for li, (W, b) in enumerate(layers):
        z = h @ bf16(W).astype(np.float64).T + b
        zs.append(z)
        if li < 3:
            h = bf16(silu(z).astype(np.float32)).astype(np.float64)
            acts.append(h)
    y = zs[-1]
    d = np.zeros_like(y)
    d[:, :OUT] = 2.0 * (y[:, :OUT] - t) / rows
    d = bf16(d.astype(np.float32)).astype(np.float64)
    loss = float(np.sum((y[:, :OUT] - t) ** 2) / rows)
    grads = [None] * 4
    for li in range(3, -1, -1):
        W, b = layers[li]
        gW = d.T @ acts[li]
        gb = d.sum(axis=0)
        grads[li] = (gW, gb)
        if li > 0:
            dh = d @ bf16(W).astype(np.float64)
            d = bf16((dh * dsilu(zs[li - 1])).astype(np.float32)).astype(np.float64)
    return grads, loss


def test_mfma_gemm_layout_and_transposes():
    banner("bf16 MFMA GEMM vs numpy (all transposition variants)")
    from avbd_amd.sim import SimulationContext
    ctx = SimulationContext(dt=1 / 60, solver_iters=1)
    ctx.add_particles(np.zeros((1, 3)), mass=np.ones(1))
    ctx.build_graph()
    rng = np.random.default_rng(0)
    M, N, K = 48, 32, 64
    A = bf16(rng.normal(size=(M, K)))
    B = bf16(rng.normal(size=(K, N)))
    for ta in (False, True):
        for tb in (False, True):
            if (ta, tb) == (True, True):
                continue
            C = ctx.mlp_gemm_test(A, B, ta, tb)
            want = A.astype(np.float64) @ B.astype(np.float64)
            err = np.abs(C - want).max() / np.abs(want).max()
            banner(f"  ta={ta} tb={tb}: rel err {err:.2e}")
            assert err < 1e-5
    # the strip kernel of the forward products (weights stored out x in, N = 128 or 16)
    for M, N, K in ((64, 128, 128), (80, 16, 128), (32, 128, 32)):
        A = bf16(rng.normal(size=(M, K)))
        B = bf16(rng.normal(size=(K, N)))
        C = ctx.mlp_gemm_test(A, B, False, True)
        want = A.astype(np.float64) @ B.astype(np.float64)
        err = np.abs(C - want).max() / np.abs(want).max()
        banner(f"  strip kernel M={M} N={N} K={K}: rel err {err:.2e}")
        assert err < 1e-5


def test_mlp_gradients_match_numpy():
    banner("MLP forward/backward vs numpy restatement")
    from avbd_amd.sim import SimulationContext
    ctx = SimulationContext(dt=1 / 60, solver_iters=1)
    ctx.add_particles(np.zeros((1, 3)), mass=np.ones(1))
    ctx.build_graph()
    ctx.mlp_init(7)
    rng = np.random.default_rng(1)
    X = rng.normal(size=(100, IN)).astype(np.float32)
    T = rng.normal(size=(100, OUT)).astype(np.float32)
    norm = np.concatenate([X.mean(0), X.std(0) + 1e-3, T.mean(0), T.std(0) + 1e-3]).astype(np.float32)
    ctx.mlp_set_normalization(norm)
    p = ctx.mlp_params()
    g, loss = ctx.mlp_forward_backward(X, T)
    ref, ref_loss = reference_grads(p, X, T)
    banner(f"  loss gpu {loss:.6f} numpy {ref_loss:.6f}")
    assert loss == pytest.approx(ref_loss, rel=1e-3)
    off = 0
    for li, (o, i) in enumerate(SHAPES):
        gW = g[off:off + o * i].reshape(o, i)
        off += o * i
        gb = g[off:off + o]
        off += o
        rW, rb = ref[li]
        eW = np.linalg.norm(gW - rW) / max(np.linalg.norm(rW), 1e-12)
        eb = np.linalg.norm(gb - rb) / max(np.linalg.norm(rb), 1e-12)
        banner(f"  layer {li}: |dW| rel err {eW:.2e}, |db| rel err {eb:.2e}")
        assert eW < 2e-2 and eb < 2e-2


def test_training_and_warm_started_solver():
    """Record (features, targets) with the plain solver on small dropped cubes,
    train on the device, then step a held-out cube warm-started and plain to
    the same residual target: the network's loss falls, every step records a
    prediction (with the incremental-potential fallback counted), both runs
    stay together, and the iteration counts of the two are reported."""
    banner("warm start: record, train, evaluate")
    from avbd_amd import scenes
    from avbd_amd import warm_start as W
    from avbd_amd.sim import Simulation, SimulationContext
    scs = W.training_scenes(3, seed=1, n_min=5, n_max=7)
    X, T = W.generate(scs, steps=30, tol=1e-2, max_iters=200, keep=1.0, log=banner)
    assert X.shape[1] == IN and T.shape[1] == OUT and np.isfinite(X).all() and np.isfinite(T).all()
    ctx = SimulationContext(dt=1 / 60, solver_iters=1)
    ctx.add_particles(np.zeros((1, 3)), mass=np.ones(1))
    ctx.build_graph()
    ctx.mlp_init(0)
    ctx.mlp_set_normalization(W.normalization(X, T))
    sel = np.random.default_rng(2).choice(X.shape[0], 4096, replace=False)
    _, loss0 = ctx.mlp_forward_backward(X[sel], T[sel])
    ctx.mlp_train(X, T, 8, 512, 1e-3, 0)
    _, loss = ctx.mlp_forward_backward(X[sel], T[sel])
    banner(f"  {X.shape[0]} rows, loss on a fixed sample {loss0:.4f} -> {loss:.4f}")
    assert loss < 0.7 * loss0
    params = ctx.mlp_params()

    sc = scenes.dropped_cube(n=6, seed=77, height=0.3)
    plain = Simulation(sc, residual_target=(1e-2, 200, 5))
    warm = Simulation(sc, residual_target=(1e-2, 200, 5))
    plain.setup()
    warm.setup()
    warm.ctx.mlp_set_params(params)
    warm.ctx.set_warm_start(True)
    plain.update(40)
    warm.update(40)
    sp, sw = plain.ctx.stats(), warm.ctx.stats()
    banner(f"  iterations plain {sp.iterations_total} warm {sw.iterations_total}; "
           f"predictions {sw.warm_start_predictions}, fallbacks {sw.warm_start_fallbacks}")
    assert sw.warm_start_predictions == 40 and sp.warm_start_predictions == 0
    xp, xw = plain.positions(), warm.positions()
    assert np.isfinite(xw).all()
    assert np.abs(xw - xp).max() < 0.05 * bbox(xp)


def bbox(x):
    return float(np.max(x.max(axis=0) - x.min(axis=0)))


def test_batched_warm_start_matches_single_scenes():
    """Warm start over a batch of scenes: the per-scene incremental-potential
    sums (block- and wavefront-level, blocks that straddle two scenes
    included) choose each scene's start as a run of that scene alone does."""
    banner("warm start: batch vs single scenes")
    from avbd_amd import scenes
    from avbd_amd import warm_start as W
    from avbd_amd.sim import Simulation
    params = W.load()
    sc = scenes.cube_batch(n_scenes=4, seed=9, n_min=4, n_max=7, iters=8, steps=6)

    def run(s):
        sim = Simulation(s, lanes_per_vertex=8, block_size=128)
        sim.setup()
        sim.ctx.mlp_set_params(params)
        sim.ctx.set_warm_start(True)
        sim.update(6)
        return sim

    b = run(sc)
    xb = b.positions()
    sb = b.ctx.stats()
    assert sb.warm_start_predictions == 6 * len(sc.meshes)
    off, fallbacks = 0, 0
    for m in sc.meshes:
        one = run(scenes.Scene(name="one", meshes=[m], iters=sc.iters, steps=sc.steps))
        xs = one.positions()
        n = xs.shape[0]
        err = np.abs(xb[off:off + n] - xs).max() / bbox(xs)
        assert err < 1e-5, err
        fallbacks += one.ctx.stats().warm_start_fallbacks
        off += n
    banner(f"  {len(sc.meshes)} scenes: batch fallbacks {sb.warm_start_fallbacks}, single runs {fallbacks}")
    assert sb.warm_start_fallbacks == fallbacks


def test_warm_start_on_the_32_cube_at_its_workload():
    """The learned warm start at its workload: the 32^3 dropped cube (35,937
    vertices), FP64 state, every step iterated to a relative force residual
    of 1e-4, the committed network, 24 steps from the drop (free fall, the
    impact and the first steps on the ground).  Every step predicts; the
    prediction is kept at the step length whose incremental-potential change
    is the most negative, and the inertial start is kept exactly when no
    length lowers it; every step meets the target; the warm run stays with
    the plain one and needs fewer iterations in total (the committed network
    saves about 7 % here, most of it on the hardest contact step)."""
    banner("warm start at its workload: 32^3 cube, residual 1e-4")
    from avbd_amd import scenes
    from avbd_amd import warm_start as W
    from avbd_amd.sim import Simulation
    params = W.load()
    sc = scenes.dropped_cube(n=32)
    tol, budget, K, steps = 1e-4, 40000, 10, 24
    runs = {}
    for warm in (False, True):
        sim = Simulation(sc, fp64_state=True, residual_target=(tol, budget, K), lanes_per_vertex=8, block_size=64,
                         gather_batch=1)
        sim.setup()
        if warm:
            sim.ctx.mlp_set_params(params)
            sim.ctx.set_warm_start(True)
        its, used = [], 0
        for k in range(steps):
            sim.update(1)
            st = sim.ctx.stats()
            its.append(st.last_step_iterations)
            assert st.residual_rel <= tol * 1.01, (warm, k, st.residual_rel)
            if warm:
                ipd, step = sim.ctx.warm_start_decision()
                best = ipd[0].min()
                if best < 0.0:
                    assert step[0] == (1.0, 0.5, 0.25)[int(np.argmin(ipd[0]))], (k, ipd, step)
                    used += 1
                else:
                    assert step[0] == 0.0, (k, ipd, step)
        st = sim.ctx.stats()
        assert st.steps_at_budget == 0
        if warm:
            assert st.warm_start_predictions == steps
            assert st.warm_start_fallbacks == steps - used
        runs[warm] = (sim.positions(), its, used)
    xp, ip, _ = runs[False]
    xw, iw, used = runs[True]
    banner(f"  iterations plain {sum(ip)} warm {sum(iw)} (gain {sum(ip) / sum(iw):.3f}); "
           f"prediction kept in {used} of {steps} steps; per step plain {ip} warm {iw}")
    assert np.abs(xw - xp).max() < 1e-3 * bbox(xp)
    assert sum(iw) < sum(ip)


@pytest.mark.parametrize("rows", [1, 15, 17, 64, 65, 1000, 4097, 8200])
def test_mlp_gradients_at_the_edges_of_the_row_chunks(rows):
    """The gradient kernel stages 64 rows at a time and splits the rows over
    at most 64 chunks: one row, around one padded strip, around one stage,
    a ragged last chunk, and chunks of more than one stage (4,097 and 8,200).
    The numpy restatement rounds the same operands to bf16; a value of dZ or H
    that falls on a rounding boundary flips by one bf16 ulp (2^-8), which the
    2 % bound per layer covers as in the test above."""
    banner(f"gradients, {rows} rows")
    from avbd_amd.sim import SimulationContext
    ctx = SimulationContext(dt=1 / 60, solver_iters=1)
    ctx.add_particles(np.zeros((1, 3)), mass=np.ones(1))
    ctx.build_graph()
    ctx.mlp_init(3)
    rng = np.random.default_rng(rows)
    X = rng.normal(size=(rows, IN)).astype(np.float32)
    T = rng.normal(size=(rows, OUT)).astype(np.float32)
    grads, loss = ctx.mlp_forward_backward(X, T)
    want, want_loss = reference_grads(ctx.mlp_params(), X, T)
    got, _ = unpack(np.concatenate([grads, np.zeros(2 * IN + 2 * OUT, np.float32)]))
    assert abs(loss - want_loss) <= 5e-3 * want_loss
    for (W, b), (gW, gb) in zip(got, want):
        assert np.linalg.norm(W - gW) <= 0.02 * np.linalg.norm(gW) + 1e-12
        assert np.linalg.norm(b - gb) <= 0.02 * np.linalg.norm(gb) + 1e-12
    again, _ = ctx.mlp_forward_backward(X, T)
    assert np.array_equal(grads, again)   # sums in a fixed order
