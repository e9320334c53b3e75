"""Cost-model MLP: the CPU oracle's analytic gradient is pinned by finite
differences (CPU); the hand-written HIP forward/backward/SGD kernels are
checked against the oracle (GPU, float32 tolerance rtol 1e-4 / atol 1e-6)."""
import numpy as np
import pytest

import mlp_oracle as mo

I, H1, H2 = 24, 64, 64


def _data(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(n, I))
    t = np.sin(x[:, 0]) + 0.3 * x[:, 1] * x[:, 2] - 0.1 * x[:, 3]
    return x, t


def test_oracle_gradient_matches_finite_differences():
    x, t = _data(40, 1)
    p = mo.init(I, H1, H2, seed=2, dtype=np.float64)
    g = mo.grad(p, x, t, I, H1, H2)
    rng = np.random.default_rng(3)
    idx = rng.choice(p.size, 60, replace=False)
    eps = 1e-6
    for k in idx:
        pp, pm = p.copy(), p.copy()
        pp[k] += eps
        pm[k] -= eps
        fd = (mo.loss(pp, x, t, I, H1, H2) - mo.loss(pm, x, t, I, H1, H2)) / (2 * eps)
        assert abs(fd - g[k]) <= 1e-6 + 1e-4 * abs(fd), (k, fd, g[k])


def test_oracle_closed_form_linear_case():
    """With ReLUs active and one hidden unit path, dL/db3 = 2 mean(y - t)."""
    x, t = _data(16, 4)
    p = mo.init(I, H1, H2, seed=5, dtype=np.float64)
    y, _ = mo.forward(p, x, I, H1, H2)
    g = mo.grad(p, x, t, I, H1, H2)
    assert np.isclose(g[-1], 2 * np.mean(y - t))


@pytest.mark.gpu
def test_gpu_forward_and_gradient_match_oracle():
    import torch
    from jacquard_amd.costmodel import MLP
    x, t = _data(1000, 6)
    p = mo.init(I, H1, H2, seed=7)
    m = MLP(params=p.copy())
    xd = torch.from_numpy(x.astype(np.float32)).cuda()
    td = torch.from_numpy(t.astype(np.float32)).cuda()
    y = torch.zeros(1000, dtype=torch.float32, device="cuda")
    m.forward_raw(xd, 1000, y)
    y_ref, _ = mo.forward(p.astype(np.float64), x.astype(np.float32).astype(np.float64), I, H1, H2)
    assert np.allclose(y.cpu().numpy(), y_ref, rtol=1e-4, atol=1e-5)
    from jacquard_amd import _native as N
    ws = torch.zeros(int(N.hip().jq_mlp_workspace_floats(I, H1, H2, 1000)),
                     dtype=torch.float32, device="cuda")
    loss = torch.zeros(1, dtype=torch.float32, device="cuda")
    m.train_step_raw(xd, td, 1000, 0.0, ws, loss)
    g_ref = mo.grad(p.astype(np.float64), x.astype(np.float32).astype(np.float64),
                    t.astype(np.float32).astype(np.float64), I, H1, H2)
    g = m.grads.cpu().numpy()
    assert np.allclose(g, g_ref, rtol=1e-3, atol=1e-6)
    assert np.isclose(loss.item(), mo.loss(p.astype(np.float64), x, t, I, H1, H2), rtol=1e-4)
    # an SGD step moves the parameters by exactly -lr * grad
    before = m.params.cpu().numpy().copy()
    m.train_step_raw(xd, td, 1000, 0.5, ws, loss)
    assert np.allclose(m.params.cpu().numpy(), before - 0.5 * m.grads.cpu().numpy(),
                       rtol=0, atol=1e-6)


@pytest.mark.gpu
def test_gpu_training_reduces_loss():
    from jacquard_amd.costmodel import MLP
    x, t = _data(5000, 8)
    m = MLP(seed=1)
    hist = m.fit(x, np.exp(t), epochs=60, lr=0.05, batch=512)
    assert hist[-1] < 0.5 * hist[0]


@pytest.mark.gpu
def test_learned_costs_against_heuristic():
    """The model trained on the batched kernel's own partition timings
    predicts held-out partition latency better than the reference heuristic
    (boomerang stages + 3, best linear fit), and the block assignment built
    from its predictions does not run slower than the heuristic's."""
    from helpers import design
    from jacquard_amd import costmodel as CM
    nl, comp = design("cm", level_split=4, seed=2, gates=300000, depth=48, dffs=20000,
                      inputs=256, outputs=128, geometric_p=0.3, invert_prob=0.5)
    W, G = 12, 2
    X, y, med = CM.training_set(comp, [W, 10, 8], G, 16)
    assert len(y) >= 5000
    s0 = comp.flatten(W)
    f0 = s0.part_features()
    truth = np.array([med[(m, i)] for (m, _b, i, _o, _l) in s0.parts.tolist()])
    h = f0[:, 0] + 3
    a, b = np.polyfit(h, truth, 1)
    mape_h = float(np.mean(np.abs(a * h + b - truth) / truth))
    model = CM.MLP(seed=1)
    model.fit(X, y, epochs=150, lr=0.05, batch=4096)
    mape_l = float(np.mean(np.abs(model.predict(f0) - truth) / truth))
    r = CM.compare_assignments(comp, W, G, {
        "reference": None, "learned": CM.stage_costs(comp, s0, model.predict(f0))},
        repeats=3, cycles=32)
    print(f"MAPE heuristic {mape_h:.3f} learned {mape_l:.3f}; us/cycle {r}", flush=True)
    assert mape_l < mape_h
    assert r["learned"] <= 1.03 * r["reference"]


@pytest.mark.gpu
def test_learned_merge_and_assignment_beat_the_heuristic():
    """On a script whose blocks run several partitions per major stage (12
    blocks for ~40 partitions per stage, as the 16M-gate workload runs about
    4.6), the learned model's merge decision plus its block assignment run
    faster than the heuristic assignment by more than the run-to-run spread
    of either, over 5 interleaved repeats; the simulated values of the
    merged design stay exact (checked against the oracle)."""
    import oracle
    from helpers import design
    from jacquard_amd import batched as B
    from jacquard_amd import costmodel as CM
    from jacquard_amd import stimulus
    nl, comp = design("cm", level_split=4, seed=2, gates=300000, depth=48, dffs=20000,
                      inputs=256, outputs=128, geometric_p=0.3, invert_prob=0.5)
    W, G = 12, 2
    costs, model, info = CM.learn_costs(comp, W, G)
    merged, mcosts, minfo = CM.learned_merge(comp, model, W, groups=G)
    assert merged is not comp and minfo["pairs_kept"] > 0
    spread = {}
    r = CM.compare_assignments(comp, W, G, {"heuristic": None, "learned+merge": (merged, mcosts)},
                               repeats=5, cycles=32, spread=spread)
    gain = r["heuristic"] - r["learned+merge"]
    print(f"us/cycle {r}, spread {spread}, merge {minfo}", flush=True)
    assert gain > max(spread["heuristic"], spread["learned+merge"]), (r, spread)
    # exact values: lanes of the merged, learned-assignment script against
    # the oracle on the original script
    s = merged.flatten(W, costs=mcosts)
    s0 = comp.flatten(W)
    seeds, probs, cyc = np.array([5, 9], np.uint32), np.array([0.2, 0.4]), np.array([24, 17])
    run = B.BatchedRun(s, seeds, probs, cyc, groups=1)
    out = run.run()
    for lane in range(2):
        st = stimulus.build_states(s0, int(cyc[lane]), seed=int(seeds[lane]), p=float(probs[lane]))
        oracle.run(s0, st, int(cyc[lane]))
        want = B.plain_observations(s0, st, int(cyc[lane]), run.obs_lits)
        assert np.array_equal(out[lane], want)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(1, 1, 1), (32, 64, 64), (17, 33, 5), (24, 16, 49), (16, 48, 64)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 300])
def test_gpu_dimensions_off_the_matrix_tiles(dims, n):
    """Layer widths and batch sizes below, at and past the 16-wide tiles and
    the 64-sample workgroups: padding adds nothing.  A unit's sum has at most
    64 products, so FP32 rounding stays below 64 * 2**-24 < 4e-6 of the sum
    of their magnitudes; the bounds leave room for the layers behind it and
    for sums that nearly cancel."""
    import torch
    from jacquard_amd import _native as N
    from jacquard_amd.costmodel import MLP
    i, h1, h2 = dims
    rng = np.random.default_rng(100 * n + i)
    x = rng.normal(size=(n, i)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    p = mo.init(i, h1, h2, seed=9).astype(np.float32)
    p += (0.05 * rng.normal(size=p.size)).astype(np.float32)
    m = MLP(params=p.copy(), i=i, h1=h1, h2=h2)
    xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    y = torch.full((n + 8,), 7.0, dtype=torch.float32, device="cuda")
    m.forward_raw(xd, n, y)
    p64, x64, t64 = (a.astype(np.float64) for a in (p, x, t))
    y_ref, _ = mo.forward(p64, x64, i, h1, h2)
    assert np.allclose(y[:n].cpu().numpy(), y_ref, rtol=1e-4, atol=1e-5)
    assert (y[n:] == 7.0).all(), "outputs past the batch"
    ws = torch.zeros(int(N.hip().jq_mlp_workspace_floats(i, h1, h2, n)),
                     dtype=torch.float32, device="cuda")
    loss = torch.zeros(1, dtype=torch.float32, device="cuda")
    m.train_step_raw(xd, td, n, 0.25, ws, loss)
    g_ref = mo.grad(p64, x64, t64, i, h1, h2)
    scale = np.abs(g_ref).max()
    assert np.allclose(m.grads.cpu().numpy(), g_ref, rtol=1e-3, atol=1e-5 * scale)
    assert np.allclose(m.params.cpu().numpy(), p64 - 0.25 * g_ref, rtol=1e-4,
                       atol=1e-5 * max(scale, 1))
    assert np.isclose(loss.item(), mo.loss(p64, x64, t64, i, h1, h2), rtol=1e-4)


@pytest.mark.gpu
def test_a_partition_takes_as_long_first_in_its_block_as_elsewhere():
    """Profiled ticks are the partition's own: flattened for several block
    counts, the partitions that lead their block in one placement and follow
    another in the next take as long in both.  A first-layer gather is about
    a quarter of a partition here, so ticks that hold it in one place only
    would differ by that; 10% leaves room for colder caches behind a
    barrier."""
    from helpers import design
    from jacquard_amd import costmodel as CM
    nl, comp = design("cm", level_split=4, seed=2, gates=300000, depth=48, dffs=20000,
                      inputs=256, outputs=128, geometric_p=0.3, invert_prob=0.5)
    seen = {}
    for W in (12, 10, 8, 6):
        s, ticks = CM.profile_batched(comp, W, 2, 18)
        block = None
        for (m, b, i, _o, _l), v in zip(s.parts.tolist(), np.median(ticks[2:], 0).tolist()):
            seen.setdefault((m, i), ([], []))[int((m, b) == block)].append(v)
            block = (m, b)
    ratio = [np.median(first) / np.median(later) for first, later in seen.values()
             if first and later]
    print(f"{len(ratio)} partitions, first in the block / elsewhere: {np.median(ratio):.3f}",
          flush=True)
    assert len(ratio) >= 30
    assert abs(np.median(ratio) - 1) < 0.1


class _Profiled:
    """Stands for a script with one partition per row of `parts`."""

    def __init__(self, parts):
        self.parts = np.array([(m, b, i, 0, 0) for m, b, i in parts], np.uint64)
        self.num_parts = len(parts)

    def part_features(self):
        return np.arange(self.num_parts * I, dtype=np.float32).reshape(-1, I)


def test_training_set_is_the_measured_ticks(monkeypatch):
    """Every sample is the ticks that were measured, whichever partition came
    first in its block, and the medians are theirs."""
    from jacquard_amd import costmodel as CM
    s = {2: _Profiled([(0, 0, 0), (0, 0, 1), (0, 1, 2), (1, 0, 0)]),
         1: _Profiled([(0, 0, 2), (0, 0, 0), (0, 0, 1), (1, 0, 0)])}
    rng = np.random.default_rng(5)
    ticks = {W: rng.integers(100, 900, (6, 4)).astype(np.float64) for W in s}
    ticks[2][:, [0, 2, 3]] += 2000  # the first of each block takes longer
    ticks[1][:, [0, 3]] += 2000
    monkeypatch.setattr(CM, "profile_batched", lambda comp, W, *a, **kw: (s[W], ticks[W]))
    X, y, med = CM.training_set(None, [2, 1], 1, 4, skip=2)
    assert X.shape == (32, I)
    assert np.array_equal(y, np.concatenate([ticks[W][2:].reshape(-1) for W in (2, 1)]))
    for key, a, b in (((0, 0), 0, 1), ((0, 1), 1, 2), ((0, 2), 2, 0), ((1, 0), 3, 3)):
        assert med[key] == np.median([np.median(ticks[2][2:, a]), np.median(ticks[1][2:, b])])


def test_learned_merge_takes_a_model_that_the_caller_fitted(monkeypatch):
    """A model with its training set kept (train_x, train_y) and nothing else
    is refitted on the trial design's measured ticks."""
    from jacquard_amd import costmodel as CM

    class Design:
        def __init__(self, n):
            self.n = n

        def flatten_shared(self, blocks):
            return _Profiled([(0, k % blocks, k) for k in range(self.n)])

        def parts_per_stage(self):
            return [self.n]

        def endpoint_counts(self):
            return [[2] * self.n]

        def merged(self, pairs):
            return Design(self.n - len(pairs)), np.ones(len(pairs), bool)

    class Model:
        train_x, train_y = np.zeros((3, I), np.float32), np.ones(3)

        def predict(self, f):
            return np.arange(10.0, 10.0 + len(f))

        def fit(self, x, y, **kw):
            self.fitted = y

    measured = np.full((6, 2), 4000.0)
    monkeypatch.setattr(CM, "profile_batched",
                        lambda comp, W, *a, **kw: (comp.flatten_shared(W), measured))
    model = Model()
    design, costs, info = CM.learned_merge(Design(4), model, 2, groups=1, sample_cycles=4)
    assert design.n == 2 and info["merged"] == 2 and info["refit_samples"] == 8
    assert np.array_equal(model.fitted, [1.0] * 3 + [4000.0] * 8)


def test_a_trial_is_one_launch(monkeypatch):
    """batched_us_per_cycle times the one launch it makes: its run-to-run
    spread, which a gain has to exceed, is that of single launches."""
    from types import SimpleNamespace
    from jacquard_amd import batched, costmodel as CM
    calls = []

    class Run:
        def __init__(self, script, seeds, probs, cycles, obs_lits, groups):
            self.n = len(seeds)

        def prepare(self):
            calls.append("prepare")

        def reset(self):
            calls.append("reset")

        def launch(self):
            calls.append("launch")

    class Event:
        def __init__(self, enable_timing):
            pass

        def record(self):
            calls.append("event")

        def elapsed_time(self, end):
            return 1.6

    cuda = SimpleNamespace(synchronize=lambda: None, Event=Event)
    monkeypatch.setattr(batched, "BatchedRun", Run)
    monkeypatch.setattr(CM, "_torch", lambda: SimpleNamespace(cuda=cuda))
    assert CM.batched_us_per_cycle(None, 2, cycles=16) == pytest.approx(100.0)
    assert calls == ["prepare", "event", "launch", "event"]


def _fma(a, b, c):
    """float32 a * b + c with one rounding: the product is exact in float64,
    and a sum rounded to odd there rounds to float32 as the exact one does."""
    p, c = np.asarray(a, np.float64) * np.asarray(b, np.float64), np.asarray(c, np.float64)
    s = np.asarray(p + c)
    v = s - p
    err = (p - (s - v)) + (c - v)
    even = (s.view(np.int64) & 1) == 0
    s = np.where((err != 0) & even, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s)
    return s.astype(np.float32)


def _chain(acc, a, b):
    """acc + a[0] b[0] + a[1] b[1] + .. in that order, one rounding each."""
    for x, y in zip(a, b):
        acc = _fma(x, y, acc)
    return acc


def _in_order(p, x, t, i, h1, h2, lr):
    """Forward, gradients, step and loss in float32 with every sum in the
    order of its index, gradients per 64 samples and then over those."""
    cut = np.cumsum([h1 * i, h1, h2 * h1, h2, h2])
    w1, b1, w2, b2, w3, b3 = np.split(p, cut)
    w1, w2 = w1.reshape(h1, i), w2.reshape(h2, h1)
    n, zero = len(x), np.float32(0)

    def layer(a, w, b):
        return _chain(np.broadcast_to(b, (n, len(b))), a.T[:, :, None], w.T[:, None, :])

    a1 = np.maximum(layer(x, w1, b1), zero)
    a2 = np.maximum(layer(a1, w2, b2), zero)
    y = layer(a2, w3[None], b3)[:, 0]
    e = y - t
    dy = np.float32(2) * e / np.float32(n)
    d2 = np.where(a2 > 0, dy[:, None] * w3, zero)
    d1 = _chain(np.zeros((n, h1), np.float32), d2.T[:, :, None], w2[:, None, :])
    d1 = np.where(a1 > 0, d1, zero)
    g, loss = np.zeros(len(p), np.float32), zero
    for s in range(0, n, 64):
        k = slice(s, s + 64)

        def outer(a, b):
            return _chain(np.zeros((a.shape[1], b.shape[1]), np.float32), a[k, :, None],
                          b[k, None, :]).reshape(-1)
        one = np.ones((n, 1), np.float32)
        g = g + np.concatenate([outer(d1, x), outer(d1, one), outer(d2, a1), outer(d2, one),
                                outer(a2, dy[:, None]), outer(dy[:, None], one)])
        loss = loss + outer((e * e)[:, None], one)[0]
    return y, g, _fma(np.float32(-lr), g, p), loss / np.float32(n)


def test_fma_rounds_once():
    """Halfway cases and products below float32's range, against the exact
    sum."""
    from fractions import Fraction
    rng = np.random.default_rng(1)
    a = np.float32(rng.normal(size=400)) * np.float32(2.0) ** rng.integers(-80, 20, 400)
    b = np.float32(rng.normal(size=400)) * np.float32(2.0) ** rng.integers(-80, 20, 400)
    c = np.where(rng.random(400) < 0.5, -(a * b).astype(np.float32), np.float32(1)).astype(np.float32)
    a, b = a.astype(np.float32), b.astype(np.float32)
    a[0], b[0], c[0] = 1 + 2.0 ** -12, 1 + 2.0 ** -12, 1  # tie to even in two roundings
    for x, y, z, r in zip(a.tolist(), b.tolist(), c.tolist(), _fma(a, b, c).tolist()):
        exact = Fraction(x) * Fraction(y) + Fraction(z)
        near = [np.nextafter(np.float32(r), np.float32(d)) for d in (-np.inf, np.inf)]
        assert all(abs(exact - Fraction(r)) <= abs(exact - Fraction(float(q))) for q in near)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,n", [((24, 64, 64), 128), ((17, 33, 5), 71)])
@pytest.mark.parametrize("scale", [1.0, 1e-20])
def test_gpu_sums_run_in_the_order_of_their_index(dims, n, scale):
    """Every output bit of the matrix-instruction kernels is that of loops
    over the summed index with one rounding a product, on whole tiles and off
    them, and with products below the normal range of float32."""
    import torch
    from jacquard_amd import _native as N
    from jacquard_amd.costmodel import MLP
    i, h1, h2 = dims
    rng = np.random.default_rng(n)
    x = (scale * rng.normal(size=(n, i))).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    p = mo.init(i, h1, h2, seed=9).astype(np.float32)
    p += (0.05 * rng.normal(size=p.size)).astype(np.float32)
    p[:h1 * i] *= np.float32(scale)
    p[h1 * i:h1 * i + h1] *= np.float32(scale * scale)
    y, g, step, loss = _in_order(p, x, t, i, h1, h2, 0.25)
    m = MLP(params=p.copy(), i=i, h1=h1, h2=h2)
    xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    yd = torch.zeros(n, dtype=torch.float32, device="cuda")
    m.forward_raw(xd, n, yd)
    ws = torch.zeros(int(N.hip().jq_mlp_workspace_floats(i, h1, h2, n)),
                     dtype=torch.float32, device="cuda")
    ld = torch.zeros(1, dtype=torch.float32, device="cuda")
    m.train_step_raw(xd, td, n, 0.25, ws, ld)
    assert np.array_equal(yd.cpu().numpy(), y)
    assert np.array_equal(m.grads.cpu().numpy(), g)
    assert np.array_equal(m.params.cpu().numpy(), step)
    assert ld.item() == loss
