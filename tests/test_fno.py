"""Learned surrogate (FNO): the FP64 numpy reference is pinned on the CPU
(finite differences, brute-force DFTs), then the HIP forward and backward
kernels are checked against it and the trained network against the plain
solver and the no-network baselines (GPU tests).

Bars: HIP forward / gradient vs FP64 reference within BF16 product
precision (relative L2 <= 2e-2 per parameter group); numpy gradient vs
central differences <= 1e-6 relative.
"""
import numpy as np
import pytest

from oracle import fno_ref as R


def tiny_shapes():
    return R.Shapes(n_theta=8, n_phi=16, width=3, modes_theta=2, modes_phi=3, layers=2)


def rand_problem(s, batch, seed, scale=0.5):
    rng = np.random.default_rng(seed)
    flat = rng.normal(0, scale, s.n_params())
    x = rng.normal(0, 1, (batch, s.T, s.P, R.N_IN))
    t = rng.normal(0, 1, (batch, s.T, s.P, R.N_OUT))
    return flat, x, t


def brute_spectral(x, Rc, s):
    """Spectral convolution by explicit double sums (no FFT)."""
    B, T, P, C = x.shape
    tt = np.arange(T)[:, None]
    pp = np.arange(P)[None, :]
    y = np.zeros_like(x)
    ks = [k if k < s.Mt // 2 else k - s.Mt for k in range(s.Mt)]
    for kk, k in enumerate(ks):
        for m in range(s.Mp):
            e = np.exp(-2j * np.pi * (k * tt / T + m * pp / P))
            X = np.einsum("btpc,tp->bc", x, e)
            Y = X @ Rc[kk, m]
            w = (1.0 if m == 0 else 2.0) / (T * P)
            y += w * np.real(np.einsum("bo,tp->btpo", Y, np.conj(e)))
    return y


def test_reference_spectral_matches_brute_force():
    s = tiny_shapes()
    rng = np.random.default_rng(1)
    x = rng.normal(0, 1, (2, s.T, s.P, s.C))
    Rc = rng.normal(0, 1, (s.Mt, s.Mp, s.C, s.C)) + 1j * rng.normal(0, 1, (s.Mt, s.Mp, s.C, s.C))
    y, _ = R.spectral(x, Rc, s)
    assert np.allclose(y, brute_spectral(x, Rc, s), rtol=1e-12, atol=1e-12)


def test_reference_gradient_finite_differences():
    s = tiny_shapes()
    flat, x, t = rand_problem(s, 2, seed=2)
    loss, g, _ = R.loss_and_grad(flat, x, t, s)
    rng = np.random.default_rng(3)
    idx = rng.choice(flat.size, 40, replace=False)
    # include the first and last entries of every group boundary region
    idx = np.unique(np.concatenate([idx, [0, flat.size - 1, flat.size - 3]]))
    eps = 1e-6
    for i in idx:
        fp, fm = flat.copy(), flat.copy()
        fp[i] += eps
        fm[i] -= eps
        num = (R.loss_and_grad(fp, x, t, s)[0] - R.loss_and_grad(fm, x, t, s)[0]) / (2 * eps)
        assert abs(num - g[i]) <= 1e-6 * max(1e-3, abs(num)) + 1e-9, (i, num, g[i])


def test_reference_gelu_grad():
    z = np.linspace(-4, 4, 101)
    num = (R.gelu(z + 1e-6) - R.gelu(z - 1e-6)) / 2e-6
    assert np.allclose(num, R.gelu_grad(z), atol=1e-8)


# ---- GPU ------------------------------------------------------------------------

GPU_CFG = dict(n_theta=32, n_phi=128, width=8, modes_theta=4, modes_phi=4, layers=2, window=4, max_batch=2)


def group_slices(s):
    C, L = s.C, s.L
    out, o = [], 0
    def add(name, n):
        nonlocal o
        out.append((name, slice(o, o + n)))
        o += n
    add("lift W", R.N_IN * C)
    add("lift b", C)
    for l in range(L):
        add("W%d" % l, C * C)
        add("b%d" % l, C)
        add("R%d" % l, s.Mt * s.Mp * 2 * C * C)
    add("Q", C * R.N_OUT)
    add("q", R.N_OUT)
    return out


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.fixture
def model():
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    m = FnoSurrogate(**GPU_CFG)
    yield m
    m.close()


@pytest.mark.gpu
def test_gpu_forward_matches_reference(model):
    s = R.Shapes.of(model.config)
    flat, x, _ = rand_problem(s, 2, seed=5, scale=0.3)
    model.set_params(flat.astype(np.float32))
    out = model.forward(x.astype(np.float32))
    ref, _, _ = R.forward(flat.astype(np.float32).astype(np.float64), x.astype(np.float32).astype(np.float64), s)
    assert rel(out, ref) <= 2e-2, rel(out, ref)


@pytest.mark.gpu
def test_gpu_gradient_matches_reference(model):
    s = R.Shapes.of(model.config)
    flat, x, t = rand_problem(s, 2, seed=6, scale=0.3)
    f32 = flat.astype(np.float32)
    model.set_params(f32)
    loss, g = model.gradient(x.astype(np.float32), t.astype(np.float32))
    rl, rg, _ = R.loss_and_grad(f32.astype(np.float64), x.astype(np.float32).astype(np.float64),
                                t.astype(np.float32).astype(np.float64), s)
    assert abs(loss - rl) <= 1e-2 * rl
    for name, sl in group_slices(s):
        assert rel(g[sl], rg[sl]) <= 2e-2, (name, rel(g[sl], rg[sl]))


# shapes served by the fused layer kernel (P = 64 RT, C = 16 CT, 2 Mp = 16 JT)
FUSED_CFG = dict(n_theta=32, n_phi=128, width=16, modes_theta=4, modes_phi=8, layers=3, window=4, max_batch=2)


@pytest.mark.gpu
def test_gpu_fused_layers_match_reference():
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    m = FnoSurrogate(**FUSED_CFG)
    s = R.Shapes.of(m.config)
    flat, x, t = rand_problem(s, 2, seed=8, scale=0.25)
    f32 = flat.astype(np.float32)
    m.set_params(f32)
    x32, t32 = x.astype(np.float32), t.astype(np.float32)
    out = m.forward(x32)
    ref, _, _ = R.forward(f32.astype(np.float64), x32.astype(np.float64), s)
    assert rel(out, ref) <= 2e-2, rel(out, ref)
    loss, g = m.gradient(x32, t32)
    rl, rg, _ = R.loss_and_grad(f32.astype(np.float64), x32.astype(np.float64), t32.astype(np.float64), s)
    assert abs(loss - rl) <= 1e-2 * rl
    for name, sl in group_slices(s):
        assert rel(g[sl], rg[sl]) <= 2e-2, (name, rel(g[sl], rg[sl]))
    m.close()


# The fused backward kernel at the corners of its shapes: every n_phi with one
# and two channel and mode tiles, a single layer (the projection's and the
# lift's gradients meet in one kernel), one grid row per block and, with more
# rows than blocks (768 of 512), an uneven walk.
@pytest.mark.gpu
@pytest.mark.parametrize("n_theta,n_phi,width,modes_theta,modes_phi,layers,batch", [
    (32, 128, 32, 4, 8, 2, 1),
    (32, 128, 16, 4, 16, 1, 2),
    (16, 256, 16, 4, 8, 1, 1),
    (16, 256, 32, 8, 16, 3, 3),
    (48, 256, 32, 3, 8, 2, 1),
    (8, 512, 32, 2, 16, 2, 1),
    (8, 512, 16, 4, 16, 2, 3),
    (256, 128, 16, 4, 8, 2, 3),
])
def test_gpu_fused_backward_shapes(n_theta, n_phi, width, modes_theta, modes_phi, layers, batch):
    from soap_bubble_simulation_amd import _lib as L
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    m = FnoSurrogate(n_theta=n_theta, n_phi=n_phi, width=width, modes_theta=modes_theta, modes_phi=modes_phi,
                     layers=layers, window=4, max_batch=batch)
    assert m.kernel_paths() & L.FNO_PATH_FUSED_ROWS
    s = R.Shapes.of(m.config)
    flat, x, t = rand_problem(s, batch, seed=31, scale=0.25)
    f32, x32, t32 = flat.astype(np.float32), x.astype(np.float32), t.astype(np.float32)
    m.set_params(f32)
    rl, rg, _ = R.loss_and_grad(f32.astype(np.float64), x32.astype(np.float64), t32.astype(np.float64), s)
    for _ in range(2):                      # the second call starts from used buffers
        loss, g = m.gradient(x32, t32)
        assert abs(loss - rl) <= 1e-2 * rl
        for name, sl in group_slices(s):
            assert rel(g[sl], rg[sl]) <= 2e-2, (name, rel(g[sl], rg[sl]))
    m.close()


@pytest.mark.gpu
def test_gpu_fused_activation_gradient_precision():
    """The activation's derivative in the fused backward pass, in FP32: with
    no spectral weights, no layer-0 matrix, a layer-1 identity and a
    projection of ones, every channel's layer-0 bias gradient is one factor
    (the same in all channels) times gelu'(bias).  In FP32 the derivative is
    off by at most 1.4e-7 and the sums by 2e-7 of up to 1.13."""
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    m = FnoSurrogate(n_theta=32, n_phi=128, width=32, modes_theta=4, modes_phi=8, layers=2, window=4, max_batch=1)
    s = R.Shapes.of(m.config)
    sl = dict(group_slices(s))
    rng = np.random.default_rng(4)
    worst = 0.0
    for _ in range(8):
        flat = np.zeros(s.n_params(), np.float32)
        b = rng.uniform(-5.0, 5.0, s.C).astype(np.float32)
        b[0] = 0.0                                  # gelu'(0) = 1/2 exactly
        flat[sl["b0"]] = b
        flat[sl["W1"]] = np.eye(s.C, dtype=np.float32).ravel()
        flat[sl["Q"]] = 1.0
        m.set_params(flat)
        x = rng.normal(0, 1, (1, s.T, s.P, R.N_IN)).astype(np.float32)
        t = np.full((1, s.T, s.P, R.N_OUT), 100.0, np.float32)
        g = m.gradient(x, t)[1][sl["b0"]].astype(np.float64)
        want = R.gelu_grad(b.astype(np.float64))
        worst = max(worst, float(np.abs(0.5 * g / g[0] - want).max()))
    m.close()
    print("activation gradient: max error %.2e" % worst)
    assert worst <= 4e-7


@pytest.mark.gpu
@pytest.mark.parametrize("width,modes_phi,layers", [(32, 16, 3), (16, 8, 2), (32, 8, 1)])
def test_gpu_inference_at_256_columns_keeps_fp32(width, modes_phi, layers):
    """n_phi = 256 keeps its activations between layers in FP32 and forms the
    lift in FP32, in inference as in training: the loss against the inference
    output is zero, where 16-bit activations put the two 1e-3 apart."""
    from soap_bubble_simulation_amd import _lib as L
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    m = FnoSurrogate(n_theta=32, n_phi=256, width=width, modes_theta=8, modes_phi=modes_phi, layers=layers, window=4,
                     max_batch=2)
    assert m.kernel_paths() == L.FNO_PATH_FUSED_ROWS | L.FNO_PATH_LIFT_DFT | L.FNO_PATH_FUSED_THETA
    s = R.Shapes.of(m.config)
    flat, x, _ = rand_problem(s, 2, seed=12, scale=0.25)
    f32, x32 = flat.astype(np.float32), x.astype(np.float32)
    m.set_params(f32)
    out = m.forward(x32)
    ref, _, _ = R.forward(f32.astype(np.float64), x32.astype(np.float64), s)
    print("n_phi 256 inference: rel", rel(out, ref))
    assert rel(out, ref) <= 2e-2, rel(out, ref)
    assert m.gradient(x32, out)[0] == 0.0
    m.close()


@pytest.mark.gpu
def test_gpu_train_step_reduces_loss(model):
    s = R.Shapes.of(model.config)
    rng = np.random.default_rng(7)
    x = rng.normal(0, 1, (2, s.T, s.P, R.N_IN)).astype(np.float32)
    # a smooth target the network can fit: a fixed linear map of the inputs
    t = np.stack([0.5 * x[..., 0] - 0.2 * x[..., 2], 0.3 * x[..., 1] + 0.1], axis=-1).astype(np.float32)
    losses = [model.train_step(x, t, lr=3e-3) for _ in range(60)]
    assert losses[-1] < 0.2 * losses[0], (losses[0], losses[-1])


# ---- surrogate on a foam: online training, judge, fallback, baselines ------------

SMALL = dict(n_theta=64, n_phi=128, width=16, modes_theta=8, modes_phi=8, layers=4, window=8, max_batch=4)


def small_foam(nb, seed, **grid):
    from soap_bubble_simulation_amd import workloads as W
    from soap_bubble_simulation_amd.foam import FoamBubble, FoamDrainage, foam_params
    T, P = grid.get("n_theta", 64), grid.get("n_phi", 128)
    d = W.foam_batch(nb, seed=seed, lat=(T, T))
    bubbles = [FoamBubble(**{**x, "n_phi": P}) for x in d]
    fm = FoamDrainage(foam_params(), bubbles)
    h = W.foam_noise(fm.offsets, [T * P] * nb, [b.h0 for b in bubbles], seed=seed + 1)
    fm.set_fields(W.ff_exact(h))
    return fm


@pytest.fixture(scope="module")
def trained():
    """A small surrogate trained online on plain-solver windows (module-wide)."""
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    m = FnoSurrogate(**SMALL)
    losses = []
    for traj in range(6):
        fm = small_foam(4, 100 + 7 * traj)
        losses.extend(m.train_foam(fm, 24, 1e-3))
        fm.close()
    yield m, np.array(losses)
    m.close()


@pytest.mark.gpu
def test_surrogate_features_match_state(trained):
    m, _ = trained
    fm = small_foam(2, 31)
    x = m.features(fm, 0, 2)
    h, g = fm.fields()
    sx, _ = m.scales()
    for k in range(2):
        hk = fm.split(h)[k]
        assert np.allclose(x[k, ..., 0], (hk / hk.mean() - 1.0) / sx, rtol=1e-4, atol=1e-4)
        th = np.arange(64) * np.pi / 63
        assert np.allclose(x[k, :, 0, 2], np.sin(th), atol=1e-6)
        assert np.all(x[k, ..., 3] == x[k, 0, 0, 3]) and np.all(x[k, ..., 4] == x[k, 0, 0, 4])
        assert np.all(x[k, ..., 5:7] == 0.0)    # no previous window: no increment
        assert np.isfinite(x[k, ..., 7]).all() and np.all(x[k, [0, -1], :, 7] == 0.0)   # one plain step


@pytest.mark.gpu
def test_surrogate_training_converges(trained):
    _, losses = trained
    # every trajectory starts with a large transient window; compare steady windows
    steady = losses.reshape(6, 24)[:, 4:]
    assert np.isfinite(losses).all()
    assert steady[-1].mean() < 0.5 * steady[0, :4].mean() or steady[-1].mean() < 0.05


@pytest.mark.gpu
def test_network_beats_extrapolation_on_held_out_bubbles(trained):
    """What the trained network gains over the method without it, on bubbles
    it never saw, from the same state after a burn-in of plain windows:

    * open loop (every window accepted), its trajectory stays far closer to
      the plain solver's than linear extrapolation of the previous increment
      (the network's input, which it corrects) does;
    * judged at the benchmark tolerance (1e-3), it is accepted several times
      as often as extrapolation and keeps h within the 1 % bar.  Judged
      extrapolation falls back to exact plain steps in most windows, and the
      one-step judge does not see smooth errors, so its trajectory error is
      the smaller one: that comparison is reported, not asserted."""
    from soap_bubble_simulation_amd import _lib as L
    m, _ = trained
    K, windows, burn = SMALL["window"], 8, 4

    def start():
        fm = small_foam(4, 999)
        fm.step(burn * K)
        return fm

    ref = start()
    h0 = ref.fields()[0]
    ref.step(windows * K)
    h_ref = ref.fields()[0]
    ref.close()
    inc = np.linalg.norm(h_ref - h0)
    res = {}
    for name, pred in (("network", L.PREDICT_NETWORK), ("extrapolate", L.PREDICT_EXTRAPOLATE)):
        for tol in (1e9, 1e-3):
            fm = start()
            st = m.advance_foam(fm, windows, tol=tol, predictor=pred)
            h = fm.fields()[0]
            res[name, tol] = dict(increment=float(np.linalg.norm(h - h_ref) / inc),
                                  h=float(np.linalg.norm(h - h_ref) / np.linalg.norm(h_ref)),
                                  accepted=int(st.accepted))
            fm.close()
    print("held-out, %d bubble-windows: %s" % (4 * windows, res))
    assert res["network", 1e9]["increment"] < 0.1 * res["extrapolate", 1e9]["increment"]
    assert res["network", 1e-3]["accepted"] >= 3 * max(1, res["extrapolate", 1e-3]["accepted"])
    assert res["network", 1e-3]["h"] <= 1e-2


@pytest.mark.gpu
def test_judge_fallback_is_exact_and_counted(trained):
    """With a tolerance no prediction meets, every window falls back to K
    plain steps from h(t): the state equals the plain solver's bit for bit."""
    from soap_bubble_simulation_amd import _lib as L
    m, _ = trained
    fm, ref = small_foam(4, 555), small_foam(4, 555)
    st = m.advance_foam(fm, 3, tol=1e-30, predictor=L.PREDICT_NETWORK)
    ref.step(3 * SMALL["window"])
    assert st.windows == 3 and st.bubble_windows == 12 and st.fallbacks == 12 and st.accepted == 0
    assert np.array_equal(fm.fields()[0], ref.fields()[0])


@pytest.mark.gpu
def test_judge_accepts_and_tracks_plain_solver(trained):
    from soap_bubble_simulation_amd import _lib as L
    m, _ = trained
    fm, ref = small_foam(4, 556), small_foam(4, 556)
    h_start = fm.fields()[0]
    st = m.advance_foam(fm, 10, tol=1e-3, predictor=L.PREDICT_NETWORK)
    ref.step(10 * SMALL["window"])
    assert st.accepted + st.fallbacks == st.bubble_windows == 40
    assert st.max_residual >= 0.0
    h_s, h_r = fm.fields()[0], ref.fields()[0]
    err = np.linalg.norm(h_s - h_r) / np.linalg.norm(h_r)
    print("accepted %d / %d, rel-L2 h %.3e, increment %.3e" % (
        st.accepted, st.bubble_windows, err, np.linalg.norm(h_s - h_r) / np.linalg.norm(h_r - h_start)))
    assert err <= 1e-2          # <= 1 % relative L2 on h


# ---- the benchmark network shape (256 x 512, width 32, 16 x 16 modes, 4 layers) ----

C4_CFG = dict(n_theta=256, n_phi=512, width=32, modes_theta=16, modes_phi=16, layers=4, window=16, max_batch=2)


def scaled_params(s, seed, spectral_std=0.1):
    """Parameters at fan-in scales, spectral weights large enough that the
    spectral path carries about as much of the output as the pointwise one."""
    rng = np.random.default_rng(seed)
    C = s.C
    parts = [rng.normal(0, 1 / np.sqrt(R.N_IN), R.N_IN * C), rng.normal(0, 0.1, C)]
    for _ in range(s.L):
        parts += [rng.normal(0, 1 / np.sqrt(C), C * C), rng.normal(0, 0.1, C),
                  rng.normal(0, spectral_std, s.Mt * s.Mp * 2 * C * C)]
    parts += [rng.normal(0, 1 / np.sqrt(C), C * R.N_OUT), rng.normal(0, 0.1, R.N_OUT)]
    return np.concatenate(parts).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 2])
def test_gpu_benchmark_shape_matches_reference(batch):
    """The network of the surrogate benchmarks: inference forward (lift
    folded into the first phi DFT, fused theta stage at 32 theta modes,
    fused row kernel at n_phi 512 and width 32) and the training forward +
    backward, against the FP64 reference."""
    from soap_bubble_simulation_amd import _lib as L
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    m = FnoSurrogate(**C4_CFG)
    paths = m.kernel_paths()
    assert paths == (L.FNO_PATH_FUSED_ROWS | L.FNO_PATH_FUSED_THETA | L.FNO_PATH_LIFT_DFT
                     | L.FNO_PATH_WAVE_ROWS), paths
    s = R.Shapes.of(m.config)
    f32 = scaled_params(s, seed=20 + batch)
    m.set_params(f32)
    rng = np.random.default_rng(30 + batch)
    x32 = rng.normal(0, 1, (batch, s.T, s.P, R.N_IN)).astype(np.float32)
    t32 = rng.normal(0, 0.3, (batch, s.T, s.P, R.N_OUT)).astype(np.float32)
    out = m.forward(x32)
    ref, _, _ = R.forward(f32.astype(np.float64), x32.astype(np.float64), s)
    print("benchmark shape, batch %d: forward rel-L2 %.2e" % (batch, rel(out, ref)))
    assert rel(out, ref) <= 2e-2, rel(out, ref)
    loss, g = m.gradient(x32, t32)
    rl, rg, _ = R.loss_and_grad(f32.astype(np.float64), x32.astype(np.float64), t32.astype(np.float64), s)
    assert abs(loss - rl) <= 1e-2 * rl
    worst = 0.0
    for name, sl in group_slices(s):
        worst = max(worst, rel(g[sl], rg[sl]))
        assert rel(g[sl], rg[sl]) <= 2e-2, (name, rel(g[sl], rg[sl]))
    print("benchmark shape, batch %d: worst gradient group rel-L2 %.2e" % (batch, worst))
    m.close()


@pytest.mark.gpu
def test_judged_foam_at_benchmark_shape():
    """The batched judge at the surrogate benchmark's network and grid
    (64 bubbles of 256 x 512, four 16-bubble chunks): every bubble-window is
    either accepted or falls back, and with a tolerance no prediction meets
    the foam ends bit-identical to the plain solver."""
    from soap_bubble_simulation_amd import _lib as L
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    cfg = dict(C4_CFG, max_batch=16)
    m = FnoSurrogate(**cfg)
    m.set_scales(0.05, 1e-3)
    grid = dict(n_theta=256, n_phi=512)
    fm, ref = small_foam(64, 77, **grid), small_foam(64, 77, **grid)
    st = m.advance_foam(fm, 2, tol=1e-30, predictor=L.PREDICT_NETWORK)
    ref.step(2 * cfg["window"])
    assert st.windows == 2 and st.bubble_windows == 128
    assert st.fallbacks == 128 and st.accepted == 0
    assert np.array_equal(fm.fields()[0], ref.fields()[0])
    st = m.advance_foam(fm, 2, tol=1e-3, predictor=L.PREDICT_IDENTITY)
    assert st.accepted + st.fallbacks == st.bubble_windows == 128
    assert st.max_residual >= 0.0
    fm.close()
    ref.close()
    m.close()


@pytest.mark.gpu
def test_judged_foam_full_benchmark_size():
    """The full surrogate benchmark foam (1024 bubbles of 256 x 512, 1.3e8
    cells, sixteen 64-bubble network chunks): with a tolerance no prediction
    meets, every bubble-window falls back and the foam ends bit-identical to
    the plain solver; with the identity predictor every bubble-window is
    accounted as accepted or fallen back."""
    from soap_bubble_simulation_amd import _lib as L
    from soap_bubble_simulation_amd.surrogate import FnoSurrogate
    cfg = dict(C4_CFG, max_batch=64)
    m = FnoSurrogate(**cfg)
    m.set_scales(0.05, 1e-3)
    grid = dict(n_theta=256, n_phi=512)
    fm, ref = small_foam(1024, 78, **grid), small_foam(1024, 78, **grid)
    assert fm.info()["cells"] >= 1024 * 256 * 512
    st = m.advance_foam(fm, 2, tol=1e-30, predictor=L.PREDICT_NETWORK)
    ref.step(2 * cfg["window"])
    assert st.windows == 2 and st.bubble_windows == 2048
    assert st.fallbacks == 2048 and st.accepted == 0
    assert np.array_equal(fm.fields()[0], ref.fields()[0])
    st = m.advance_foam(fm, 1, tol=1e-3, predictor=L.PREDICT_IDENTITY)
    assert st.accepted + st.fallbacks == st.bubble_windows == 1024
    fm.close()
    ref.close()
    m.close()
