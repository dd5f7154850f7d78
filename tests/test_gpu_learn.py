"""GPU tests of the learned warm start: the MFMA network and the training kernels against the numpy
specification (oracle/mlp_oracle.py), the features, the fallback, the warm-started step against
the CPU oracle's warm-started step, and what a trained network gains."""
import os
import sys

import numpy as np
import pytest

import meshgen as M
import phybs_amd as P
from oracle import mlp_oracle as MO
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

SCALES = np.array([0.5, 1.0, 2.0, 0.3, 0.7, 1.5, 0.8], np.float32)


def say(*a):
    print("[gpu-test]", *a, flush=True)
    sys.stdout.flush()


def bar(twist=30.0, jitter=0.01):
    rest, tets = M.bar(4, 4, 16, 0.05)
    mask = M.clamp_x0(rest)
    x0 = M.twisted_state(rest, 4, 4, 16, 0.05, twist, jitter, 1)
    return rest, tets, mask, x0


def model(seed=3):
    p = MO.init_params(seed)
    p[1152:1216] = 0.1  # nonzero first-layer biases
    return p


def test_mlp_forward_matches_spec():
    rest, tets, mask, _ = bar()
    say("MFMA forward vs numpy")
    s = P.Solver(rest, tets, mask, P.default_params())
    s.learn_set_model(model(), SCALES)
    f = np.random.default_rng(0).normal(0, 1, (1000, 18)).astype(np.float32)
    got = s.learn_forward(f)
    ref, _ = MO.forward(model(), SCALES, f)
    err = np.abs(got - ref)
    scale = np.abs(ref).max()
    say("max err", err.max(), "of", scale, "fraction above 1e-4 x max:", np.mean(err > 1e-4 * scale))
    # FP32 accumulation order differs; a hidden activation whose BF16 rounding flips moves an
    # output by ~1e-3 of its scale, which happens for a small fraction of samples
    assert err.max() <= 1e-2 * scale
    assert np.mean(err > 1e-4 * scale) <= 0.01
    s.close()


def test_mlp_loss_and_gradient_match_spec():
    rest, tets, mask, _ = bar()
    say("training gradient vs numpy")
    s = P.Solver(rest, tets, mask, P.default_params())
    s.learn_set_model(model(), SCALES)
    rng = np.random.default_rng(1)
    f = rng.normal(0, 1, (777, 18)).astype(np.float32)
    t = rng.normal(0, 1, (777, 3)).astype(np.float32)
    loss, g = s.learn_loss_grad(f, t)
    lref, gref = MO.loss_grad(model(), SCALES, f, t)
    say("loss", loss, lref, "grad rel err", np.linalg.norm(g - gref) / np.linalg.norm(gref))
    assert loss == pytest.approx(lref, rel=1e-5)
    assert np.linalg.norm(g - gref) <= 1e-3 * np.linalg.norm(gref)
    s.close()


@pytest.mark.parametrize("n", [1, 16, 17, 64, 65, 16385])
def test_training_at_the_edges_of_its_tiles(n):
    """One sample, one wave's 16 and one more, a workgroup's 64 and one more, one more than 256
    workgroups take in a first tile: loss and gradient against numpy, and after one Adam step the
    forward pass (which reads the arranged BF16 weights) against numpy on the read-back parameters.
    Tolerances as in the tests above; where a hidden activation's BF16 rounding flips, a sample's
    share (1 / n) of loss and gradient moves by up to 1 and 2 per cent."""
    rest, tets, mask, _ = bar()
    say("training tiles", n)
    s = P.Solver(rest, tets, mask, P.default_params())
    s.learn_set_model(model(), SCALES)
    rng = np.random.default_rng(n)
    f = rng.normal(0, 1, (n, 18)).astype(np.float32)
    t = rng.normal(0, 1, (n, 3)).astype(np.float32)
    loss, g = s.learn_loss_grad(f, t)
    lref, gref = MO.loss_grad(model(), SCALES, f, t)
    say("loss", loss, lref, "grad rel err", np.linalg.norm(g - gref) / np.linalg.norm(gref))
    assert loss == pytest.approx(lref, rel=1e-5 + 1e-2 / n)
    assert np.linalg.norm(g - gref) <= (1e-3 + 2e-2 / n) * np.linalg.norm(gref)
    s.learn_collect(n)
    s.learn_add_samples(f, t)
    s.learn_train(1, batch=n, lr=1e-2, seed=3)
    p, sc = s.learn_get_model()
    assert not np.array_equal(p, model())
    out, ref = s.learn_forward(f), MO.forward(p, sc, f)[0]
    assert np.abs(out - ref).max() <= 1e-2 * np.abs(ref).max()
    s.close()


@pytest.mark.parametrize("n", [65, 700, 5003])
def test_no_activation_rounds_to_the_other_side(n):
    """Loss and gradient against 64 bits with the same BF16 roundings (of inputs, weights and hidden
    activations, these from their exact values).  Every activation rounds as the exact one, so what is
    left is FP32 rounding of deltas and sums, about 2e-7; taken 5 times as large.  One activation on
    the other side would cost about 5e-3 / n."""
    say("training against 64 bits", n)
    rest, tets, mask, _ = bar()
    s = P.Solver(rest, tets, mask, P.default_params())
    s.learn_set_model(model(), SCALES)
    inv = (np.float32(1) / SCALES).astype(np.float64)
    p = list(zip(*MO.unpack(model(), np.float64)))
    for seed in range(3):
        rng = np.random.default_rng(seed)
        f = rng.normal(0, 1, (n, 18)).astype(np.float32)
        t = rng.normal(0, 1, (n, 3)).astype(np.float32)
        loss, g = s.learn_loss_grad(f, t)
        bf = lambda a: MO.bf16(a.astype(np.float32)).astype(np.float64)
        h, z = [bf(f * np.repeat(inv[:6], 3))], []
        for k, (w, b) in enumerate(p):
            z.append(h[-1] @ bf(w) + b)
            h.append(bf(MO.silu(z[-1])) if k < 3 else z[-1])
        diff = h[-1] - t * inv[6]
        lref, d, gref = (diff ** 2).mean(), 2 * diff / diff.size, []
        for k in range(3, -1, -1):
            gref = [(h[k].T @ d).reshape(-1), d.sum(0)] + gref
            if k:
                d = (d @ bf(p[k][0]).T) * MO.dsilu(z[k - 1])
        gref = np.concatenate(gref)
        err = np.linalg.norm(g - gref) / np.linalg.norm(gref)
        say("loss", loss, lref, "grad rel err %.2e" % err)
        assert loss == pytest.approx(lref, rel=1e-6) and err <= 1e-6
    s.close()


def adjacency(nn, tets):
    nb = [set() for _ in range(nn)]
    for t in tets:
        for a in t:
            for b in t:
                if a != b:
                    nb[a].add(int(b))
    off = np.zeros(nn + 1, np.int64)
    adj = []
    for n in range(nn):
        adj += sorted(nb[n])
        off[n + 1] = len(adj)
    return off, np.array(adj, np.int64)


def test_features_match_spec():
    rest, tets, mask, x0 = bar()
    say("features")
    h = float(np.float32(0.03))
    s = P.Solver(rest, tets, mask, P.default_params(precision=P.FP64))
    s.set_positions(x0)
    for _ in range(2):
        s.step()
    got = s.learn_features()
    x = s.positions(f64=True)
    v = s.velocities()[0]
    off, adj = adjacency(len(rest), tets)
    ref = MO.features(x, v, rest, h, np.float32([0.0, -9.8, 0.0]).astype(np.float64), off, adj, mask)
    scale = np.abs(ref).max(axis=0) + 1e-30
    err = (np.abs(got - ref) / scale).max()
    say("max rel err (per feature scale)", err)
    assert err <= 1e-5  # velocities cross the boundary as FP32
    assert not got[mask != 0].any()
    s.close()


def test_rejected_guess_leaves_the_plain_trajectory_unchanged():
    rest, tets, mask, x0 = bar()
    say("fallback: a far-off guess is rejected, the trajectory is bitwise the plain one")
    bad_scales = SCALES.copy()
    bad_scales[6] = 1e3  # outputs of order 1 become displacements of order 1 km
    runs = []
    for warm in (False, True):
        s = P.Solver(rest, tets, mask, P.default_params(precision=P.FP64, relgrad_tol=1e-4, max_iterations=5000))
        s.set_positions(x0)
        if warm:
            s.learn_set_model(model(), bad_scales)
            s.learn_enable(True)
        st = [s.step() for _ in range(3)]
        runs.append((s.positions(f64=True), st))
        s.close()
    (xp, sp), (xl, sl) = runs
    # the far-off guess has a larger (or non-finite) gradient norm and is not used
    assert all(q.used_learned == 0 and not (q.g_learned <= q.g0_norm) for q in sl)
    assert [q.iterations for q in sp] == [q.iterations for q in sl]
    assert [q.g0_norm for q in sp] == [q.g0_norm for q in sl]
    assert np.array_equal(xp.view(np.uint64), xl.view(np.uint64))


def trained_model(rest, tets, mask, gp, seed=5, steps=12):
    """A network trained on another trajectory (seeded twist, impulses) of the same bar."""
    t = P.Solver(rest, tets, mask, gp)
    t.set_positions(M.twisted_state(rest, 4, 4, 16, 0.05, 60.0, 0.01, seed))
    t.learn_collect(steps * len(rest))
    rng = np.random.default_rng(seed)
    for k in range(steps):
        ext = np.zeros_like(rest)
        if k % 4 == 2:
            ext[rng.integers(0, len(rest), 10)] = rng.normal(0, 5.0, (10, 3))
        t.step(ext)
    t.learn_fit_scales()
    t.learn_init_model(seed)
    t.learn_train(40, batch=256, lr=3e-3, seed=seed)
    m = t.learn_get_model()
    t.close()
    return m


@pytest.mark.parametrize("net", ["trained", "random"])
def test_warm_started_step_matches_oracle(net):
    """FP64: the GPU's learned guess handed to the oracle's warm-started step (which evaluates both
    guesses' gradients and keeps the better) gives the same decision, iterations and positions,
    for a trained network (its guess is taken in some steps) and a random one (always rejected)."""
    rest, tets, mask, x0 = bar()
    say("warm-started step vs oracle,", net, "network")
    gp = P.default_params(precision=P.FP64, relgrad_tol=1e-4, max_iterations=5000)
    if net == "trained":
        params, sc = trained_model(rest, tets, mask, gp)
    else:
        params, sc = model(), SCALES.copy()
        sc[6] = 2e-3
    s = P.Solver(rest, tets, mask, gp)
    s.set_positions(x0)
    s.learn_set_model(params, sc)
    s.learn_enable(True)
    o = O.Solver(rest, tets, mask, params=O.default_params(relgrad_tol=1e-4, iterations=5000), precision=64)
    o.set_state(x=x0.astype(np.float64))
    h, mom = float(np.float32(0.03)), float(np.float32(0.2))
    used = []
    for k in range(8):
        learned, plain = s.learn_guess()
        xs, vs, vls = o.state()
        assert np.abs(plain - (xs + h * vs + mom * (vs - vls) * h)).max() <= 1e-9
        gs = s.step()
        os_ = o.step(x0=learned)
        say("step", k, "used gpu/oracle", gs.used_learned, os_.used_learned, "its", gs.iterations, os_.iterations,
            "g_l/g0 %.3f" % (gs.g_learned / gs.g0_norm))
        assert gs.used_learned == os_.used_learned
        assert gs.g0_norm == pytest.approx(os_.g0_norm, rel=1e-6)
        assert abs(gs.iterations - os_.iterations) <= 2
        assert np.abs(s.positions(f64=True) - o.state()[0]).max() <= 1e-7 * 0.8
        used.append(gs.used_learned)
    say("guess used in steps", used)
    assert (net == "trained") == any(used)
    s.close()


def test_collect_and_train_on_gpu():
    rest, tets, mask, x0 = bar()
    say("collect + train")
    s = P.Solver(rest, tets, mask, P.default_params(precision=P.FP64, relgrad_tol=1e-4, max_iterations=5000))
    s.set_positions(x0)
    nfree = int((mask == 0).sum())
    s.learn_collect(10 * nfree)
    s.step()
    v32, vl32 = s.velocities()
    s.set_velocities(v32, vl32)  # the state's velocities are now exactly these FP32 values
    s.learn_collect(10 * nfree)
    x_before = s.positions(f64=True)
    v_before = v32.astype(np.float64)
    s.step()
    x_after = s.positions(f64=True)
    assert s.learn_samples() == nfree
    f, t = s.learn_get_samples()
    # target = converged position - (x + h v + h^2 g), free nodes in node order
    h = float(np.float32(0.03))
    y = x_before + h * v_before + h * h * np.float32([0, -9.8, 0]).astype(np.float64)
    ref = (x_after - y)[mask == 0]
    assert np.abs(t - ref).max() <= 1e-6 * np.abs(ref).max() + 1e-12
    for _ in range(9):
        s.step()
    assert s.learn_samples() == 10 * nfree
    s.step()  # full: not collected
    assert s.learn_samples() == 10 * nfree
    s.learn_fit_scales()
    s.learn_init_model(5)
    loss = s.learn_train(8, batch=512, lr=3e-3, seed=2)
    say("loss per epoch", np.round(loss, 5))
    assert loss[-1] < 0.5 * loss[0]
    # the trained model's loss on the samples, through the C ABI, equals the numpy one
    p, sc = s.learn_get_model()
    lg, _ = s.learn_loss_grad(f, t)
    lo, _ = MO.loss_grad(p, sc, f, t)
    assert lg == pytest.approx(lo, rel=1e-4)
    s.close()


def bench_params(**kw):
    return P.default_params(precision=P.FP64, relgrad_tol=1e-4, max_iterations=20000, dt=1 / 30.0,
                            grav=(0.0, 0.0, -9.8), profile=[(1, 0.96), (7, 0.991), (10, 0.9995)], **kw)


def warm_run(rest, tets, mask, prm, x0, steps, mdl=None, collect=0, stride=1, seed=None, sweeps=10, warmup=0):
    """steps steps from x0 (impulses on 10 random nodes every 10th step when seed is given);
    returns (solver, stats of the steps after the warm-up)."""
    s = P.Solver(rest, tets, mask, prm)
    s.set_positions(x0)
    if collect:
        s.learn_collect(collect, stride)
    if mdl is not None:
        s.learn_set_model(*mdl)
        s.learn_enable(True)
        s.learn_set_options(sweeps, (1.0,))
    r = np.random.default_rng(seed) if seed is not None else None
    st = []
    for k in range(warmup + steps):
        ext = None
        if r is not None and k % 10 == 5:
            ext = np.zeros_like(rest)
            ext[r.integers(0, len(rest), 10)] = r.normal(0, 20, (10, 3))
        q = s.step(ext)
        if k >= warmup:
            st.append(q)
    return s, st


def test_trained_warm_start_gain():
    """What the trained network gains on the benchmark's own configuration: the 64x64x256 bar
    (6.3 M tets) sagging from rest under gravity, rel-grad 1e-4.  The network is trained on the
    plain solver's own trajectory from a held-out start (0.2 % jitter, seed 7, impulses; every
    4th free node of 30 steps, 8 M pairs), then the evaluation trajectory (from rest, no jitter)
    runs with and without the warm start (5 warm-up steps, 10 measured): the guess is used in at
    least 80 % of the steps and saves at least a quarter of the iterations, and both runs reach
    rel-grad 1e-4 in every step.  The gradient test guarantees that a worse guess is never used."""
    sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    import bench

    dims = (64, 64, 256)
    rest, tets = P.mesh_bar(*dims, 0.05)
    mask = (rest[:, 0] == 0).astype(np.int32)
    prm = bench_params()
    say("64x64x256 warm start: collecting the training trajectory")
    s = bench.collect_trajectory(P, rest, tets, mask, P.mesh_twist(rest, *dims, 0.05, 0.0, 0.002, 7), prm, 30, 7, 4,
                                 12_000_000)
    s.learn_fit_scales()
    s.learn_init_model(7)
    loss = s.learn_train(30, batch=8192, lr=2e-3, seed=7)
    mdl = s.learn_get_model()
    s.close()
    sp, stp = warm_run(rest, tets, mask, prm, rest, 10, warmup=5)
    sl, stl = warm_run(rest, tets, mask, prm, rest, 10, mdl, warmup=5, sweeps=20)
    ip = np.mean([q.iterations for q in stp])
    il = np.mean([q.iterations for q in stl])
    used = np.mean([q.used_learned for q in stl])
    say("trained: loss %.4f -> %.4f; iterations/step plain %.1f, warm-started %.1f (%.1f%% saved), guess used in "
        "%.0f%% of steps" % (loss[0], loss[-1], ip, il, 100 * (ip - il) / ip, 100 * used))
    assert loss[-1] < 0.2 * loss[0]
    assert all(q.converged and q.g_norm <= 1e-4 * q.g0_norm for q in stl + stp)
    assert used >= 0.8
    assert il <= 0.75 * ip
    xp, xl = sp.positions(f64=True), sl.positions(f64=True)
    say("|x_learned - x_plain| after 15 steps: %.2e m (bar length 12.8 m)" % np.abs(xl - xp).max())
    assert np.abs(xl - xp).max() <= 1e-4 * 12.8
    sp.close()
    sl.close()
    # the same network under the mixed mode (FP32 forces down to |g|/|g0| = 2e-4): every step
    # still converges on FP64 passes, with the warm-start decision of the FP64 run's first step
    sm, stm = warm_run(rest, tets, mask, bench_params(mixed_switch=2e-4), rest, 5, mdl, warmup=5, sweeps=20)
    assert all(q.converged and q.g_norm <= 1e-4 * q.g0_norm for q in stm)
    assert stm[0].used_learned == stl[0].used_learned
    say("mixed + warm start: iterations/step %.1f (FP64: %.1f over the same 5 steps)"
        % (np.mean([q.iterations for q in stm]), np.mean([q.iterations for q in stl[:5]])))
    sm.close()


def test_bar12x12x50_warm_start_protocol():
    """The benchmark's warm-start protocol on the 12x12x50 bar released from a 90 degree twist
    (1 % jitter, seed 11), network trained on the plain solver's trajectories from other seeds (2
    and 3, impulses).  On this bar the network does not beat the plain
    guess: its predicted corrections carry short-wavelength errors that the gradient test sees,
    and the guess is rejected in most steps.  What the test holds: every step converges to
    rel-grad 1e-4, the warm start costs at most 2 % of the plain iterations, and the trajectory
    matches the plain one to the solver's tolerance.  The iterations saved are printed."""
    dims = (12, 12, 50)
    rest, tets = M.bar(*dims, 0.05)
    mask = M.clamp_x0(rest)
    prm = bench_params()
    s, _ = warm_run(rest, tets, mask, prm, M.twisted_state(rest, *dims, 0.05, 90.0, 0.01, 2), 60,
                    collect=2_000_000, seed=2)
    q, _ = warm_run(rest, tets, mask, prm, M.twisted_state(rest, *dims, 0.05, 90.0, 0.01, 3), 60,
                    collect=1_000_000, seed=3)
    f, t = q.learn_get_samples()
    q.close()
    s.learn_add_samples(f, t)
    s.learn_fit_scales()
    s.learn_init_model(7)
    s.learn_train(30, batch=8192, lr=2e-3, seed=7)
    mdl = s.learn_get_model()
    s.close()
    x0 = M.twisted_state(rest, *dims, 0.05, 90.0, 0.01, 11)
    sp, stp = warm_run(rest, tets, mask, prm, x0, 30, warmup=1)
    sl, stl = warm_run(rest, tets, mask, prm, x0, 30, mdl, warmup=1)
    ip = np.mean([q.iterations for q in stp])
    il = np.mean([q.iterations for q in stl])
    used = np.mean([q.used_learned for q in stl])
    say("12x12x50 bar: iterations/step plain %.1f, warm-started %.1f (%.2f%% saved), guess used in %.0f%% of steps"
        % (ip, il, 100 * (ip - il) / ip, 100 * used))
    assert all(q.converged and q.g_norm <= 1e-4 * q.g0_norm for q in stl)
    assert il <= 1.02 * ip
    assert np.abs(sl.positions(f64=True) - sp.positions(f64=True)).max() <= 1e-4 * 2.5
    sp.close()
    sl.close()
