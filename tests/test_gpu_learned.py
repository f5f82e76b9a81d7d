"""GPU tests of the learned coarse step through the C ABI, against the FP64
reference in oracle/surrogate_ref.py.

* sph_mlp_train gradients (FP32 forward/backward kernels, deterministic
  reduction) equal the FP64 analytic gradient of the same batch to 1e-4
  relative norm; the loss to 1e-5.
* sph_mlp_predict (FP32 path) equals the FP64 forward to 1e-4.
* Adam steps on the GPU lower the loss of a fixed batch.
* One coarse step (network, and the SPH force held for 4 fine steps) equals
  the FP64 coarse integrator from the same state.
* The judge with a zero drift limit keeps the 4-plain-step result.
"""
import importlib.util
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ref():
    spec = importlib.util.spec_from_file_location("surrogate_ref", os.path.join(ROOT, "oracle", "surrogate_ref.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


NORM = dict(v_scale=0.1, rho_scale=1e-5, pi_scale=5e-4, acc_scale=2e4)


def _norm(pkg):
    return pkg.sph.MlpNorm(NORM["v_scale"], NORM["rho_scale"], NORM["pi_scale"], NORM["acc_scale"])


def _scene(pkg, orc, n=1500, steps=30):
    sc = pkg.scenes.dam10k()
    p0 = orc.lattice(sc.nx, sc.ny, sc.nz, sc.spacing, sc.origin, sc.jitter, sc.seed, count=sc.count)[:n].copy()
    b = pkg.sph.make_boundary(sc.lower, sc.upper)
    sim = pkg.Simulation(n, boundaries=b)
    sim.upload(p0)
    sim.step(steps)
    return sim, sc


def _cpu_pairs(state, perm, h, slots):
    """Neighbour pairs (r < h, j != i) of the given target slots, by brute force
    in float32 arithmetic on the same positions."""
    pos = state["pos"][perm, :3]
    rows_t, rows_j = [], []
    h2 = np.float32(h) * np.float32(h)
    margin = []
    for t, s in enumerate(slots):
        d = (pos[s][None, :] - pos).astype(np.float32)
        r2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]).astype(np.float32)
        near = np.nonzero((r2 < h2) & (np.arange(len(pos)) != s))[0]
        margin.append(np.min(np.abs(r2.astype(np.float64) / float(h2) - 1.0)))
        rows_t += [t] * len(near)
        rows_j += list(near)
    return np.array(rows_t), np.array(rows_j), float(np.min(margin))


def _features(ref, state, perm, slots, rows_t, rows_j, h):
    st = state[perm]
    x = st["pos"][:, :3].astype(np.float64)
    v = st["vel"][:, :3].astype(np.float64)
    rho = st["extras"][:, 0].astype(np.float64)
    p = st["extras"][:, 1].astype(np.float64)
    inv_rho = (np.float32(1.0) / st["extras"][:, 0]).astype(np.float64)
    i = np.asarray(slots)[rows_t]
    j = rows_j
    return ref.pair_features(x[i], x[j], v[i], v[j], rho[i], rho[j], p[i], p[j], inv_rho[j], float(h), NORM)


def _targets(state_now, state_later, perm, slots, sc):
    a = state_now[perm][slots]
    b = state_later[perm][slots]
    dt = np.float32(1.0) / np.float32(10000.0)
    g = np.array([0.0, np.float32(-9806.65), 0.0])
    acc = (b["vel"][:, :3].astype(np.float64) - a["vel"][:, :3]) / (4 * float(dt)) - g
    lo, hi = np.array(sc.lower, dtype=np.float32), np.array(sc.upper, dtype=np.float32)
    ok = np.ones(len(slots), dtype=bool)
    for st in (a, b):
        ps = st["pos"][:, :3]
        ok &= np.all(np.isfinite(ps), axis=1) & np.all((np.abs(ps - lo) > 1e-6) & (np.abs(ps - hi) > 1e-6), axis=1)
    tgt = np.where(ok[:, None], acc / NORM["acc_scale"], 0.0)
    return tgt, ok.astype(np.float64)


def _cluster(orc, n, seed=3):
    """n particles, each within h of every other."""
    rng = np.random.default_rng(seed)
    p = orc.particles(n)
    p["pos"][:, :3] = rng.uniform(0.0, 0.008, (n, 3)).astype(np.float32)
    p["vel"][:, :3] = rng.normal(0, 5, (n, 3)).astype(np.float32)
    return p


def test_training_gradient_matches_fp64(pkg, orc, ref, gpu_lib):
    sim, sc = _scene(pkg, orc)
    later = pkg.Simulation(sim.n, boundaries=pkg.sph.make_boundary(sc.lower, sc.upper))
    later.copy_state_from(sim)
    later.step(4)
    params = ref.init_params(7)
    params[ref.NPARAMS - 195:] += np.random.default_rng(8).normal(0, 0.05, 195).astype(np.float32)
    sim.mlp_set(params, _norm(pkg))
    first, stride = 1, 2
    res, grad = sim.mlp_train(later, first=first, stride=stride, update=False, want_grad=True)
    now = sim.download()
    lat = later.download()
    _, perm = sim.download_grid()
    slots = np.arange(first, sim.n, stride)
    h = orc.smoothing_length()
    rows_t, rows_j, margin = _cpu_pairs(now, perm, h, slots)
    assert margin > 1e-6, "fixture has a pair on the r = h boundary"
    assert res.pairs == len(rows_t) and res.targets == len(slots)
    f = _features(ref, now, perm, slots, rows_t, rows_j, h)
    tgt, w = _targets(now, lat, perm, slots, sc)
    assert res.weighted == int(w.sum())
    L, g, _ = ref.loss_and_grad(params.astype(np.float64), f, rows_t, tgt, w)
    assert res.loss == pytest.approx(L, rel=1e-5)
    assert np.linalg.norm(grad - g) <= 1e-4 * np.linalg.norm(g)
    sim.close()
    later.close()


def test_predict_fp32_matches_fp64(pkg, orc, ref, gpu_lib):
    sim, sc = _scene(pkg, orc, n=1200, steps=20)
    params = ref.init_params(11)
    sim.mlp_set(params, _norm(pkg))
    pred = sim.mlp_predict(path=0)
    now = sim.download()
    _, perm = sim.download_grid()
    slots = np.arange(sim.n)
    h = orc.smoothing_length()
    rows_t, rows_j, margin = _cpu_pairs(now, perm, h, slots)
    assert margin > 1e-6
    f = _features(ref, now, perm, slots, rows_t, rows_j, h)
    m, _ = ref.forward(params.astype(np.float64), f)
    cpu = np.zeros((sim.n, 3))
    np.add.at(cpu, rows_t, m)
    cpu_aos = np.zeros_like(cpu)
    cpu_aos[perm] = cpu
    scale = np.abs(m).sum() / len(m) * 200
    assert np.max(np.abs(pred - cpu_aos)) <= 1e-4 * scale
    sim.close()


def test_adam_lowers_loss(pkg, orc, ref, gpu_lib):
    sim, sc = _scene(pkg, orc, n=1500, steps=40)
    later = pkg.Simulation(sim.n, boundaries=pkg.sph.make_boundary(sc.lower, sc.upper))
    later.copy_state_from(sim)
    later.step(4)
    sim.mlp_set(ref.init_params(5), _norm(pkg))
    losses = [sim.mlp_train(later, lr=3e-3).loss for _ in range(60)]
    assert losses[-1] < 0.5 * losses[0]
    p, nm = sim.mlp_get()
    assert np.all(np.isfinite(p)) and nm.acc_scale == NORM["acc_scale"]
    sim.close()
    later.close()


@pytest.mark.parametrize("use_network", [False, True])
def test_coarse_step_matches_fp64_integrator(pkg, orc, ref, gpu_lib, use_network):
    sim, sc = _scene(pkg, orc, n=2000, steps=25)
    params = ref.init_params(13)
    sim.mlp_set(params, _norm(pkg))
    s0 = sim.download()
    if use_network:
        pred = sim.mlp_predict(path=1).astype(np.float64)  # the coarse step runs the MFMA kernel
        acc = NORM["acc_scale"] * pred + np.array([0.0, np.float32(-9806.65), 0.0])
    else:
        sim.rho_pres()
        sim.force()
        sf = sim.download()
        acc = sf["force"][:, :3].astype(np.float64) / sf["extras"][:, [0]].astype(np.float64)
    sim.upload(s0)
    st = sim.coarse_step(1, use_network=use_network)
    assert st.coarse_steps == 1 and st.plain_steps == 0
    got = sim.download()
    dt = float(np.float32(1.0) / np.float32(10000.0))
    x, v = ref.coarse_integrate(s0["pos"][:, :3].astype(np.float64), s0["vel"][:, :3].astype(np.float64), acc,
                                sc.lower, sc.upper, dt, float(np.float32(0.3)))
    vscale = np.abs(s0["vel"][:, :3]) + 4 * dt * np.abs(acc) + 1e-3
    # Axes whose unclamped FP64 position lies within 1e-5 of a wall may take
    # either clamp branch in float32.
    xu = s0["pos"][:, :3].astype(np.float64) + 4 * dt * s0["vel"][:, :3] + 10 * dt * dt * acc
    lo, hi = np.array(sc.lower)[None, :], np.array(sc.upper)[None, :]
    strict = (np.abs(xu - lo) > 1e-5) & (np.abs(xu - hi) > 1e-5)
    assert strict.mean() > 0.9
    assert np.all((np.abs(got["vel"][:, :3] - v) <= 2e-5 * vscale)[strict])
    assert np.all((np.abs(got["pos"][:, :3] - x) <= 1e-6)[strict])
    sim.close()


def test_judge_zero_limit_keeps_plain_result(pkg, orc, ref, gpu_lib):
    sim, sc = _scene(pkg, orc, n=2000, steps=10)
    sim.mlp_set(ref.init_params(17), _norm(pkg))
    s0 = sim.download()
    st = sim.coarse_step(3, use_network=True, judge_every=1, drift_limit=0.0, cooldown=0)
    assert st.judged == 3 and st.fallbacks == 3 and st.coarse_steps == 0 and st.plain_steps == 12
    got = sim.download()
    with pkg.Simulation(sim.n, boundaries=pkg.sph.make_boundary(sc.lower, sc.upper)) as plain:
        plain.upload(s0)
        plain.step(12)
        want = plain.download()
    assert got["pos"].tobytes() == want["pos"].tobytes() and got["vel"].tobytes() == want["vel"].tobytes()
    # cooldown: after a fallback the next coarse steps run plain.
    sim.upload(s0)
    st = sim.coarse_step(4, use_network=True, judge_every=4, drift_limit=0.0, cooldown=3)
    assert st.fallbacks == 1 and st.plain_steps == 16 and st.coarse_steps == 0
    sim.close()


def test_predict_mfma_matches_fp32(pkg, orc, ref, gpu_lib):
    """BF16 MFMA messages equal the FP32 path to BF16 accuracy, on a scene with
    more than 512 neighbour hits for some particles (hit-list wrap-around)."""
    sim, sc = _scene(pkg, orc, n=4000, steps=5)
    params = ref.init_params(19)
    params[ref.NPARAMS - 195:] += np.random.default_rng(20).normal(0, 0.05, 195).astype(np.float32)
    sim.mlp_set(params, _norm(pkg))
    p32 = sim.mlp_predict(path=0)
    _poison_predictions(sim, pkg, ref, params)
    pbf = sim.mlp_predict(path=1)
    assert np.all(np.isfinite(pbf))
    rel = np.linalg.norm(pbf - p32) / np.linalg.norm(p32)
    assert rel < 2e-2, rel
    # crowded: every particle within h of every other (hit lists longer than one LDS list)
    n = 700
    with pkg.Simulation(n) as dense:
        p = orc.particles(n)
        p["pos"][:, :3] = np.random.default_rng(1).uniform(0.0, 0.008, (n, 3)).astype(np.float32)
        dense.upload(p)
        dense.mlp_set(params, _norm(pkg))
        a = dense.mlp_predict(path=0)
        _poison_predictions(dense, pkg, ref, params)
        b = dense.mlp_predict(path=1)
        assert np.linalg.norm(b - a) / np.linalg.norm(a) < 2e-2


@pytest.mark.parametrize("sub", [1, 3])
def test_predict_mfma_every_stencil_size(pkg, orc, ref, gpu_lib, sub):
    """The message kernel at 1 and 3 cells per h (9 and 49 stencil rows, one
    lane each) matches the FP32 path to BF16 accuracy and the 2-cells-per-h
    messages up to the summation order, also where hit lists overflow."""
    sim, sc = _scene(pkg, orc, n=4000, steps=5)
    params = ref.init_params(19)
    params[ref.NPARAMS - 195:] += np.random.default_rng(20).normal(0, 0.05, 195).astype(np.float32)
    sim.mlp_set(params, _norm(pkg))
    p2 = sim.mlp_predict(path=1)
    sim.set_tuning(cells_per_h=sub)
    p32 = sim.mlp_predict(path=0)
    _poison_predictions(sim, pkg, ref, params)
    pbf = sim.mlp_predict(path=1)
    assert np.all(np.isfinite(pbf))
    assert np.linalg.norm(pbf - p32) / np.linalg.norm(p32) < 2e-2
    assert np.linalg.norm(pbf - p2) / np.linalg.norm(p2) < 1e-4
    sim.close()
    n = 700
    with pkg.Simulation(n) as dense:
        p = orc.particles(n)
        p["pos"][:, :3] = np.random.default_rng(1).uniform(0.0, 0.008, (n, 3)).astype(np.float32)
        dense.upload(p)
        dense.set_tuning(cells_per_h=sub)
        dense.mlp_set(params, _norm(pkg))
        a = dense.mlp_predict(path=0)
        _poison_predictions(dense, pkg, ref, params)
        b = dense.mlp_predict(path=1)
        assert np.linalg.norm(b - a) / np.linalg.norm(a) < 2e-2


def test_trained_network_beats_no_network(pkg, orc, gpu_lib):
    """The committed weights (trained on the GPU on 200 dam1m rollouts) predict
    the 4-step mean acceleration of held-out states better than the method
    without the network (the SPH force held over the 4 steps) and than zero."""
    import sys
    sys.path.insert(0, os.path.join(ROOT, "npr-sph_amd"))
    import train_surrogate
    params, norm, meta = train_surrogate.load_weights()
    assert meta["rollouts"] >= 200 and meta["workload"] == "dam1m"
    sph = pkg.sph
    sc = pkg.scenes.dam1m(seed=4242)  # seed not used in training
    b = sph.make_boundary(sc.lower, sc.upper)
    G = np.array([0.0, np.float32(-9806.65), 0.0])
    dt = float(np.float32(1.0) / np.float32(10000.0))
    with pkg.Simulation(sc.count, boundaries=b) as sim, pkg.Simulation(sc.count, boundaries=b) as later:
        sim.init_lattice(sph.make_lattice(**sc.lattice_args()))
        sim.step(600)
        later.copy_state_from(sim)
        later.step(4)
        sim.mlp_set(params, norm)
        pred = sim.mlp_predict(path=1).astype(np.float64)
        a, l = sim.download(), later.download()
        sim.rho_pres()
        sim.force()
        f = sim.download()
    with np.errstate(invalid="ignore", divide="ignore"):
        sph_acc = f["force"][:, :3].astype(np.float64) / f["extras"][:, [0]] - G
    tgt = (l["vel"][:, :3].astype(np.float64) - a["vel"][:, :3]) / (4 * dt) - G
    lo, hi = np.array(sc.lower, np.float32), np.array(sc.upper, np.float32)
    ok = np.all(np.isfinite(tgt), 1) & np.all(np.isfinite(sph_acc), 1)
    for st in (a, l):
        ps = st["pos"][:, :3]
        ok &= np.all((np.abs(ps - lo) > 1e-6) & (np.abs(ps - hi) > 1e-6), 1)
    A = norm.acc_scale

    def loss(p):
        return float(np.mean(np.sum((p[ok] - tgt[ok] / A) ** 2, 1)))

    l_net, l_sph, l_zero = loss(pred), loss(sph_acc / A), loss(np.zeros_like(tgt))
    assert l_net < 0.5 * l_zero and l_net < 0.1 * l_sph, (l_net, l_sph, l_zero)


def test_coarse_step_counts_every_pair(pkg, orc, gpu_lib):
    """sph_coarse_stats_t.pairs equals the number of ordered neighbour pairs
    (r < h, j != i) of the state the message pass ran on, counted by brute force
    in float32 on the CPU."""
    params = np.random.default_rng(3).normal(0, 0.05, pkg.sph.MLP_PARAMS).astype(np.float32)
    sim, sc = _scene(pkg, orc)
    with sim:
        sim.mlp_set(params, _norm(pkg))
        st = sim.download()
        stats = sim.coarse_step(1, use_network=True)
    pos = st["pos"][:, :3].astype(np.float32)
    h2 = np.float32(orc.smoothing_length()) * np.float32(orc.smoothing_length())
    total, margin = 0, np.inf
    for i in range(len(pos)):
        d = (pos[i][None, :] - pos).astype(np.float32)
        r2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]).astype(np.float32)
        r2[i] = np.inf
        total += int(np.count_nonzero(r2 < h2))
        margin = min(margin, float(np.min(np.abs(r2.astype(np.float64) / float(h2) - 1.0))))
    assert margin > 1e-6  # no pair so close to r = h that float32 rounding could decide it
    assert stats.pairs == total and total > 0


def test_repeated_rejections_keep_the_plain_trajectory(pkg, orc, ref, gpu_lib):
    """With a zero drift limit every judge rejects: after each rejection the
    cooldown runs plain steps and the next step is judged again, so no coarse
    step is ever accepted and the state equals the plain run bit for bit."""
    sim, sc = _scene(pkg, orc, n=2000, steps=10)
    sim.mlp_set(ref.init_params(23), _norm(pkg))
    s0 = sim.download()
    st = sim.coarse_step(10, use_network=True, judge_every=50, drift_limit=0.0, cooldown=2)
    # judged at 0, 3, 6, 9 (each after a 2-step cooldown)
    assert (st.judged, st.fallbacks, st.coarse_steps, st.plain_steps) == (4, 4, 0, 40)
    got = sim.download()
    with pkg.Simulation(sim.n, boundaries=pkg.sph.make_boundary(sc.lower, sc.upper)) as plain:
        plain.upload(s0)
        plain.step(40)
        want = plain.download()
    assert got["pos"].tobytes() == want["pos"].tobytes() and got["vel"].tobytes() == want["vel"].tobytes()
    # A limit no drift reaches accepts every judged step.
    sim.upload(s0)
    st = sim.coarse_step(3, use_network=True, judge_every=1, drift_limit=1e30, cooldown=2)
    assert (st.judged, st.fallbacks, st.coarse_steps, st.plain_steps) == (3, 0, 3, 0)
    sim.close()


def test_dam8m_learned_leg(pkg, orc, gpu_lib):
    """The large mixed run's learned leg at its real size: dam8m (8,000,000
    particles) after 150 steps, with the committed weights.
    * The BF16 MFMA messages (the kernel fused into the cell-sorted gather)
      equal the FP32 message path to BF16 accuracy over all particles.
    * The pairs one message pass evaluates equal the FP64 grid count of
      neighbour pairs (r < h, j != i) of that state, up to pairs within 1e-6
      of r = h, whose side float32 rounding decides.
    * Three coarse steps judged every step by 4 plain steps: each judged step
      is accepted or replaced, the drift is a finite relative figure and the
      state stays finite except the reference's own coincident-pair NaNs."""
    import sys
    sys.path.insert(0, os.path.join(ROOT, "npr-sph_amd"))
    import train_surrogate
    params, norm, _ = train_surrogate.load_weights()
    sc = pkg.scenes.dam8m()
    b = pkg.sph.make_boundary(sc.lower, sc.upper)
    ob = orc.make_boundary(sc.lower, sc.upper)
    with pkg.Simulation(sc.count, boundaries=b) as sim:
        sim.init_lattice(pkg.sph.make_lattice(**sc.lattice_args()))
        sim.step(150)
        sim.mlp_set(params, norm)
        s0 = sim.download()
        p32 = sim.mlp_predict(path=0)
        pbf = sim.mlp_predict(path=1)
        ok = np.all(np.isfinite(p32), axis=1)
        assert ok.mean() > 0.999
        assert np.array_equal(ok, np.all(np.isfinite(pbf), axis=1))
        rel = np.linalg.norm(pbf[ok] - p32[ok]) / np.linalg.norm(p32[ok])
        assert rel < 2e-2, rel
        del p32, pbf
        sim.upload(s0)
        st = sim.coarse_step(1, use_network=True, judge_every=0, drift_limit=0.0, cooldown=0)
        want, amb = orc.count_pairs(orc.pos64(s0), b=ob, margin=1e-6)
        assert want > 100 * sc.count
        assert abs(st.pairs - want) <= amb, (st.pairs, want, amb)
        sim.upload(s0)
        st = sim.coarse_step(3, use_network=True, judge_every=1, drift_limit=0.01, cooldown=0)
        assert st.judged == 3 and st.coarse_steps + st.fallbacks == 3
        assert st.plain_steps == 4 * st.fallbacks
        assert np.isfinite(st.max_drift) and 0.0 <= st.max_drift < 1.0
        m = sim.metrics(0)
        assert np.isfinite(m.mean_rho) and m.mean_rho > 1000.0
        # Non-finite particles: the reference's coincident-pair NaNs (normalize(0)
        # where corner walls clamp particles onto one point), as in 12 plain steps.
        sim.upload(s0)
        sim.step(12)
        mp = sim.metrics(0)
        assert mp.nonfinite < 1e-3 * sc.count
        assert m.nonfinite <= 2 * mp.nonfinite + 100, (m.nonfinite, mp.nonfinite)


def _count_pairs_only(ref, value):
    """A network whose message is `value` for every pair."""
    params = np.zeros(ref.NPARAMS, np.float32)
    params[-3:] = value
    return params


def _poison_predictions(sim, pkg, ref, params):
    """Leaves 10^6 per neighbour in the prediction buffer, then loads `params`:
    a target that the next pass leaves out shows."""
    sim.mlp_set(_count_pairs_only(ref, 1e6), _norm(pkg))
    sim.mlp_predict(path=0)
    sim.mlp_set(params, _norm(pkg))


def _assert_gradient_is_the_sum_over(sim, later, k):
    """The training gradient over all particles is the weighted sum of those of
    every k-th from 0 .. k-1.  Bound: each is within 1e-6 of its norm or better
    (float32 sums of some 2,048 rows, added in double)."""
    res, grad = sim.mlp_train(later, first=0, stride=1, update=False, want_grad=True)
    parts = [sim.mlp_train(later, first=i, stride=k, update=False, want_grad=True) for i in range(k)]
    for name in ("pairs", "targets", "weighted"):
        assert getattr(res, name) == sum(getattr(r, name) for r, _ in parts)
    assert res.loss * res.weighted == pytest.approx(sum(r.loss * r.weighted for r, _ in parts), rel=1e-9)
    got = grad.astype(np.float64) * res.weighted
    want = sum(g.astype(np.float64) * r.weighted for r, g in parts)
    size = sum(np.linalg.norm(g.astype(np.float64)) * r.weighted for r, g in parts)
    assert np.linalg.norm(got) > 0.0
    assert np.linalg.norm(got - want) <= 1e-6 * (np.linalg.norm(got) + size), (np.linalg.norm(got - want), np.linalg.norm(got))
    return res


@pytest.mark.parametrize("n", [513, 65535, 65536, 65601])
def test_network_takes_every_target_once(pkg, orc, ref, gpu_lib, n):
    """Targets go to the XCDs one a wave below 65,536 and in runs of 64 from
    there, to waves of 4 or (backward pass) 8 a workgroup.  Messages that count a target's
    pairs, into a buffer that held others, are the same on both paths and add up
    to the oracle's count, up to pairs that float32 rounding decides; so does what the
    16-bit pass and the training step count; the gradient is that of two halves,
    dealt in another way."""
    rng = np.random.default_rng(n)
    side = (n * 1e-6) ** (1.0 / 3.0)
    p = orc.particles(n)
    p["pos"][:, :3] = rng.uniform(0.0, side, (n, 3)).astype(np.float32)
    q = p.copy()
    q["vel"][:, :3] = rng.normal(0, 5, (n, 3)).astype(np.float32)
    bounds = (0.0,) * 3, (side,) * 3
    want, unsure = orc.count_pairs(orc.pos64(p), b=orc.make_boundary(*bounds))
    with pkg.Simulation(n, boundaries=pkg.sph.make_boundary(*bounds)) as sim, pkg.Simulation(n) as later:
        sim.upload(p)
        later.upload(q)
        counts = []
        for path in (1, 0):
            _poison_predictions(sim, pkg, ref, _count_pairs_only(ref, 1.0))
            counts.append(sim.mlp_predict(path=path))
        assert np.array_equal(counts[0], counts[1])
        assert abs(counts[0][:, 0].astype(np.float64).sum() - want) <= unsure
        sim.mlp_set(ref.init_params(3), _norm(pkg))
        res = _assert_gradient_is_the_sum_over(sim, later, 2)
        assert abs(res.pairs - want) <= unsure and res.targets == n
        assert sim.coarse_step(1, use_network=True).pairs == res.pairs


def test_training_gradient_over_several_targets_a_wave(pkg, orc, ref, gpu_lib):
    """6,144 targets of 1,535 neighbours, three to each wave of the backward
    pass: a wave moves its sums to its partial after two of them (more than
    2,048 rows) and once more at the end.  Every third and every fourth target
    alone give a wave one at most."""
    n, m = 1536, 4
    p = np.concatenate([_cluster(orc, n, seed) for seed in range(m)])
    p["pos"][:, 0] += np.repeat(0.1 * np.arange(m, dtype=np.float32), n)
    q = p.copy()
    q["vel"][:, :3] += np.random.default_rng(5).normal(0, 5, (n * m, 3)).astype(np.float32)
    with pkg.Simulation(n * m) as sim, pkg.Simulation(n * m) as later:
        sim.upload(p)
        later.upload(q)
        sim.mlp_set(ref.init_params(3), _norm(pkg))
        for k in (3, 4):
            res = _assert_gradient_is_the_sum_over(sim, later, k)
            assert res.pairs == m * n * (n - 1) and res.targets == m * n


@pytest.mark.parametrize("n", [1, 2, 16, 17, 18, 130, 193, 700])
@pytest.mark.parametrize("sub", [1, 2, 3])
def test_network_tiles(pkg, orc, ref, gpu_lib, n, sub):
    """FP32 messages and the training gradient where every particle has n - 1
    neighbours: no pair, partly filled and full 16-pair tiles, and hit lists
    that are processed before the scan ends (more than 128 hits).  Targets run
    from one to n, over one and several waves.  Bounds: a message sum of k
    terms carries at most about k float32 roundings (6e-8 each) of its terms'
    magnitude; the gradient's sums run over up to n^2 pairs."""
    rng = np.random.default_rng(n)
    params = ref.init_params(29)
    params[ref.NPARAMS - 195:] += rng.normal(0, 0.05, 195).astype(np.float32)
    p = orc.particles(n)
    p["pos"][:, :3] = rng.uniform(0.0, 0.008, (n, 3)).astype(np.float32)
    p["vel"][:, :3] = rng.normal(0, 5, (n, 3)).astype(np.float32)
    q = p.copy()
    q["vel"][:, :3] += rng.normal(0, 5, (n, 3)).astype(np.float32)
    with pkg.Simulation(n) as sim, pkg.Simulation(n) as later:
        for s, state in ((sim, p), (later, q)):
            s.set_tuning(cells_per_h=sub)
            s.upload(state)
        sim.mlp_set(params, _norm(pkg))
        pred = sim.mlp_predict(path=0)
        now = sim.download()
        _, perm = sim.download_grid()
        h = orc.smoothing_length()
        for first, stride in ((0, 1), (n - 1, 1), (n // 2, 3)):
            slots = np.arange(first, n, stride)
            rows_t, rows_j, margin = (np.zeros(0, int), np.zeros(0, int), 1.0) if n == 1 else _cpu_pairs(now, perm, h, slots)
            assert margin > 1e-6
            f = _features(ref, now, perm, slots, rows_t, rows_j, h)
            if stride == 1 and first == 0:
                m, _ = ref.forward(params.astype(np.float64), f)
                want = np.zeros((n, 3))
                np.add.at(want, rows_t, m)
                assert np.abs(pred[perm] - want).max() <= 6e-8 * n * n + 1e-6 * (np.abs(m).max() if len(m) else 0) * n
                # 16-bit operands: 2^-9 of each factor of a message's terms, which partly cancel in a sum.
                for shrink in (1.0, 1e-6, 1e30):
                    small = params.copy()
                    small[ref.NPARAMS - 195:] *= np.float32(shrink)
                    sim.mlp_set(small, _norm(pkg))
                    half = sim.mlp_predict(path=1)[perm]
                    assert np.linalg.norm(half - shrink * want) <= 2e-2 * np.linalg.norm(shrink * want)
                wild = params.copy()  # activations beyond FP16's largest saturate
                wild[:640] *= np.float32(1e7)
                sim.mlp_set(wild, _norm(pkg))
                assert np.isfinite(sim.mlp_predict(path=1)).all()
                sim.mlp_set(params, _norm(pkg))
            res, grad = sim.mlp_train(later, first=first, stride=stride, update=False, want_grad=True)
            assert res.pairs == len(rows_t) and res.targets == len(slots)
            tgt, w = _targets(now, q, perm, slots, pkg.scenes.dam10k())
            L, g, _ = ref.loss_and_grad(params.astype(np.float64), f, rows_t, tgt, w)
            assert res.loss == pytest.approx(L, rel=1e-5)
            assert np.linalg.norm(grad - g) <= 1e-5 * np.linalg.norm(g)


def test_messages_16bit_keep_first_layer_weights(pkg, orc, ref, gpu_lib):
    """First-layer weights that BF16 would all round towards zero, by 0.49 units in its
    last place: rounded so, the messages are 2.7e-3 off; what rounds at random (inputs,
    activations, W2) averages out over 129 pairs and 64 units to 5e-4."""
    n = 130
    params = ref.init_params(29)
    params[ref.NPARAMS - 195:] += np.random.default_rng(n).normal(0, 0.05, 195).astype(np.float32)
    w1 = params[:576]
    w1[:] = (w1.view(np.uint32) & 0xffff0000).view(np.float32)
    w1 += np.sign(w1) * np.float32(0.49) * np.exp2(np.floor(np.log2(np.abs(w1))) - 7).astype(np.float32)
    with pkg.Simulation(n) as sim:
        sim.upload(_cluster(orc, n))
        sim.rho_pres()
        norm = _norm(pkg)
        norm.rho_scale = float(1.3 / sim.download()["extras"][:, 0].mean())
        norm.pi_scale = float(1.0 / sim.download()["extras"][:, 1].mean()) * float(sim.download()["extras"][:, 0].mean())
        sim.mlp_set(params, norm)
        half = sim.mlp_predict(path=1).astype(np.float64)
        full = sim.mlp_predict(path=0).astype(np.float64)
    assert np.linalg.norm(half - full) <= 1.2e-3 * np.linalg.norm(full)


@pytest.mark.parametrize("z1", [-4.0, -60.0, -3e4, 1e5, 0.5])
@pytest.mark.parametrize("z2", [-5.0, -100.0, -2e4, 3.5, 700.0])
def test_messages_16bit_gelu_tails(pkg, orc, ref, gpu_lib, z1, z2):
    """16-bit messages where every activation of a layer has the same input, in
    the tails of the GELU: the training form stays at -0.00197 below -3, and an
    offset there has one sign over all pairs.  Bounds of an activation's error:
    1e-5 in the negative tail (coefficients and FP16 rounding), elsewhere the
    lookup's 2^-7 of the value; inputs beyond 65504 saturate.  The second layer
    passes the first's error on."""
    n = 34
    params = np.zeros(ref.NPARAMS, np.float32)
    params[576:640] = z1
    params[640:640 + 4096] = np.eye(64, dtype=np.float32).ravel()
    params[4736:4800] = z2
    params[4800:4992] = 1.0
    h1 = ref.gelu(min(z1, 65504.0))
    h2 = ref.gelu(min(h1 + z2, 65504.0))
    err1 = 1e-5 if z1 < -3 else abs(h1) * 2.0**-7
    err2 = 1e-5 if h1 + z2 < -3 else abs(h2) * 2.0**-7
    with pkg.Simulation(n) as sim:
        sim.upload(_cluster(orc, n))
        sim.mlp_set(params, _norm(pkg))
        got = sim.mlp_predict(path=1).astype(np.float64)
    slope = 1.0 if h1 + err1 + z2 > -3 else 0.0
    assert np.abs(got / (64 * (n - 1)) - h2).max() <= err2 + slope * err1


def test_messages_16bit_infinite_activations(pkg, orc, ref, gpu_lib):
    """A first layer that overflows to minus infinity ends in the GELU's
    negative tail, as any large negative input does."""
    n = 34
    params = np.zeros(ref.NPARAMS, np.float32)
    params[6 * 64:7 * 64] = params[576:640] = -3e38
    params[4800:4992] = 1.0
    params[640:640 + 4096] = np.eye(64, dtype=np.float32).ravel()
    params[4736:4800] = -5.0
    with pkg.Simulation(n) as sim:
        sim.upload(_cluster(orc, n))
        sim.rho_pres()
        norm = _norm(pkg)
        norm.rho_scale = float(16.0 / sim.download()["extras"][:, 0].min())
        sim.mlp_set(params, norm)
        got = sim.mlp_predict(path=1).astype(np.float64)
    assert np.abs(got / (64 * (n - 1)) - ref.gelu(-5.0)).max() <= 1e-5


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("n", [2, 34, 300])
def test_messages_16bit_show_nonfinite_inputs(pkg, orc, ref, gpu_lib, value, n):
    """A particle of non-finite velocity makes its own message and its
    neighbours' non-finite, and no other's: two clusters, one of them with it."""
    p = np.concatenate([_cluster(orc, n), _cluster(orc, n, 4)])
    p["pos"][n:, 0] += 0.1
    p["vel"][n // 2, 1] = value
    with pkg.Simulation(2 * n) as sim:
        sim.upload(p)
        sim.mlp_set(ref.init_params(31), _norm(pkg))
        half = sim.mlp_predict(path=1)
        full = sim.mlp_predict(path=0)
    assert not np.isfinite(half[:n]).any() and np.isfinite(half[n:]).all()
    assert np.array_equal(np.isfinite(half), np.isfinite(full))


@pytest.mark.parametrize("layer", ["W2", "W3"])
def test_messages_16bit_show_diverged_weights(pkg, orc, ref, gpu_lib, layer):
    """Weights that an Adam update made NaN (eps = 0 and no gradient: 0/0) in
    one layer alone make the messages NaN on both paths.  A unit whose input
    weights are zero passes 0 on, so its output weights get no gradient."""
    n = 34
    d = ref.unpack(ref.init_params(31))
    d["w3"] += np.random.default_rng(32).normal(0, 0.05, d["w3"].shape)
    if layer == "W2":
        d["w1"][:, 5] = 0.0
    else:
        d["w2"][:, 5] = 0.0
    p = _cluster(orc, n)
    q = _cluster(orc, n)
    q["vel"][:, :3] += np.random.default_rng(33).normal(0, 5, (n, 3)).astype(np.float32)
    with pkg.Simulation(n) as sim, pkg.Simulation(n) as later:
        sim.upload(p)
        later.upload(q)
        sim.mlp_set(ref.pack(d).astype(np.float32), _norm(pkg))
        sim.mlp_train(later, lr=1e-3, eps=0.0)
        got = ref.unpack(sim.mlp_get()[0])
        for name in ("w1", "b1", "w2", "b2", "w3", "b3"):
            bad = np.isnan(got[name])
            if name == layer.lower():
                assert bad[5].all() and not np.delete(bad, 5, axis=0).any()
            else:
                assert not bad.any()
        assert np.isnan(sim.mlp_predict(path=1)).all()
        assert np.isnan(sim.mlp_predict(path=0)).all()


@pytest.mark.parametrize("case", ["plain", "small", "tiny", "huge", "units", "low edge", "high edge", "outputs"])
def test_messages_16bit_any_weight_size(pkg, orc, ref, gpu_lib, case):
    """W2 and W3 of any size, beyond FP16's range and among its subnormals, in
    networks whose activations are of ordinary size: the earlier layer or the
    later one is scaled the other way.  W2 has one scale a unit where a unit's
    largest weight (half of it for 2 units in 4) leaves [2^-8, 65504], none inside it.  Bound: one
    rounding of each input to BF16, 2^-9; over 64 units and 129 pairs roundings
    average out to less."""
    n = 130
    rng = np.random.default_rng(41)
    d = ref.unpack(ref.init_params(29))
    d["w3"] += rng.normal(0, 0.05, d["w3"].shape)
    d["b1"], d["b2"] = rng.normal(0, 0.1, 64), rng.normal(0, 0.1, 64)
    one, two = {"small": (1e4, 1e-4), "tiny": (1e4, 1e-5), "huge": (1e-3, 1e7)}.get(case, (1.0, 1.0))
    d["w1"] *= one
    d["b1"] *= one
    d["w2"] *= two
    d["b2"] *= min(two * one, 1.0)
    big = np.abs(d["w2"]).max(axis=0)
    if case == "units":
        k = 10.0 ** np.linspace(-3, 3, 64)
        d["w2"] *= k
        d["b2"] *= k
        d["w3"] /= k[:, None]
    elif case == "low edge":  # half the units just above the edge, half below
        k = np.where(np.arange(64) % 4 < 2, 2.0**-7, 2.0**-8) / big * np.where(np.arange(64) % 2, 1.001, 0.999)
        d["w1"] *= 30.0
        d["b1"] *= 30.0
        d["w2"] *= k
    elif case == "high edge":
        k = np.where(np.arange(64) % 4 < 2, 131008.0, 65504.0) / big * np.where(np.arange(64) % 2, 1.001, 0.999)
        d["w1"] *= 1e-4
        d["b1"] *= 1e-4
        d["w2"] *= k
    elif case == "outputs":
        d["w3"] *= [1e-12, 1.0, 1e9]
    params = ref.pack(d).astype(np.float32)
    with pkg.Simulation(n) as sim:
        sim.upload(_cluster(orc, n))
        sim.rho_pres()
        norm = _norm(pkg)
        norm.rho_scale = float(1.3 / sim.download()["extras"][:, 0].mean())
        norm.pi_scale = float((sim.download()["extras"][:, 0] / sim.download()["extras"][:, 1]).mean())
        sim.mlp_set(params, norm)
        half = sim.mlp_predict(path=1).astype(np.float64)
        full = sim.mlp_predict(path=0).astype(np.float64)
    assert np.isfinite(full).all()
    assert (np.linalg.norm(half - full, axis=0) <= 2.0**-9 * np.linalg.norm(full, axis=0)).all()


@pytest.mark.parametrize("scale", [3e-6, 2e-5, 6e-5])
def test_messages_16bit_small_activations(pkg, orc, ref, gpu_lib, scale):
    """Activations among FP16's subnormals: the lookup takes its values' centres
    2^-20 apart, so an activation is within 2^-21 and its GELU, of slope 1/2 there, within
    2^-22 (plus the polynomial's and rounding's 2^-24).  One
    activation per unit over the range, passed on by a diagonal W3."""
    n = 34
    x = np.random.default_rng(43).uniform(-scale, scale, (2, 64))
    for row in x.astype(np.float32):
        err = np.zeros(64)
        for c in range(0, 64, 3):  # three units at a time, one an output
            params = np.zeros(ref.NPARAMS, np.float32)
            params[4736:4800] = row
            for k, u in enumerate(range(c, min(c + 3, 64))):
                params[4800 + 3 * u + k] = 1.0
            with pkg.Simulation(n) as sim:
                sim.upload(_cluster(orc, n))
                sim.mlp_set(params, _norm(pkg))
                got = sim.mlp_predict(path=1).astype(np.float64) / (n - 1)
            for k, u in enumerate(range(c, min(c + 3, 64))):
                err[u] = np.abs(got[:, k] - ref.gelu(float(row[u]))).max()
        assert err.max() <= 2.0**-22 + 2.0**-24, err.max()


@pytest.mark.parametrize("n", [64, 65, 66, 129, 256, 257, 321, 513])
def test_network_long_rows(pkg, orc, ref, gpu_lib, n):
    """All particles in one grid cell, a stencil row of n slots: rows of more
    than 64 slots are listed by the whole wave, lists of 256 (16-bit messages,
    backward pass) and 512 candidates cut them, and a second cluster in the next
    cell gives a wave a long and a short row.  Messages and gradient against FP64 as in
    test_network_tiles."""
    rng = np.random.default_rng(n)
    params = ref.init_params(29)
    params[ref.NPARAMS - 195:] += rng.normal(0, 0.05, 195).astype(np.float32)
    short = 5
    p = orc.particles(n + short)
    p["pos"][:, :3] = rng.uniform(0.0001, 0.001, (n + short, 3)).astype(np.float32)
    p["pos"][n:, 1] += 0.006
    p["vel"][:, :3] = rng.normal(0, 5, (n + short, 3)).astype(np.float32)
    q = p.copy()
    q["vel"][:, :3] += rng.normal(0, 5, (n + short, 3)).astype(np.float32)
    h = orc.smoothing_length()
    with pkg.Simulation(n + short) as sim, pkg.Simulation(n + short) as later:
        sim.upload(p)
        later.upload(q)
        sim.mlp_set(params, _norm(pkg))
        half = sim.mlp_predict(path=1)
        pred = sim.mlp_predict(path=0)
        now = sim.download()
        _, perm = sim.download_grid()
        slots = np.arange(n + short)
        rows_t, rows_j, margin = _cpu_pairs(now, perm, h, slots)
        assert margin > 1e-6
        f = _features(ref, now, perm, slots, rows_t, rows_j, h)
        m, _ = ref.forward(params.astype(np.float64), f)
        want = np.zeros((n + short, 3))
        np.add.at(want, rows_t, m)
        assert np.abs(pred[perm] - want).max() <= 6e-8 * n * n + 1e-6 * np.abs(m).max() * n
        # 16-bit: all pairs are nearly alike, so the lookups' errors (2^-7 of a value) do not average over them.
        assert np.linalg.norm(half[perm] - want) <= 2.0**-7 * np.linalg.norm(want)
        res, grad = sim.mlp_train(later, first=0, stride=1, update=False, want_grad=True)
        assert res.pairs == len(rows_t)
        tgt, w = _targets(now, q, perm, slots, pkg.scenes.dam10k())
        L, g, _ = ref.loss_and_grad(params.astype(np.float64), f, rows_t, tgt, w)
        assert res.loss == pytest.approx(L, rel=1e-5)
        assert np.linalg.norm(grad - g) <= 1e-5 * np.linalg.norm(g)
        assert sim.coarse_step(1, use_network=True).pairs == len(rows_t)
