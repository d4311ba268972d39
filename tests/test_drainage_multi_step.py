"""Several steps per launch on small grids (drainage_multi_kernel) against the
FP64 oracle and against one step per launch."""
import ctypes as C

import numpy as np
import pytest

from soap_bubble_simulation_amd import _lib as L
from soap_bubble_simulation_amd import workloads as W
from soap_bubble_simulation_amd.drainage import DrainageContext

pytestmark = pytest.mark.gpu

TFE, SURF, MARA = L.FLAG_TFE, L.FLAG_SURFACTANT, L.FLAG_MARANGONI
COPY, AVG, DIAG = L.FLAG_POLES_COPY_H, L.FLAG_POLES_AVG_GAMMA, L.FLAG_DIAG


def _params(flags, rebase=8):
    p = L.Params()
    L.check(L.lib().sf_params_cpu_default(p))
    p.flags = flags
    p.rebase_interval = rebase
    p.tfe_first_spawn = 0.0            # a front from the first step on
    p.sin_guard = 1e-4
    return p


def _fields(nt, npf, seed):
    h = W.noise_field(nt, npf, seed, rel=0.05)
    rng = np.random.default_rng(seed + 1)
    h.reshape(-1)[rng.choice(h.size, max(1, h.size // 50), replace=False)] = 9e-9      # ruptured cells
    g = np.float32(0.5 + 0.2 * rng.uniform(-1, 1, (nt, npf))).astype(np.float64)
    return W.ff_exact(h), g


# Grids: the fewest rows and columns, one row per block and rows that do not
# divide among the blocks, odd and single columns, more columns than threads.
GRIDS = [(3, 1), (3, 7), (4, 8), (7, 64), (64, 128), (128, 256), (129, 255), (300, 601), (500, 1003), (514, 1024),
         (12, 1500)]
FLAGS = [0, TFE, SURF, TFE | SURF | DIAG, SURF | COPY, MARA | SURF | AVG | DIAG, MARA, MARA | SURF | COPY | DIAG]


@pytest.mark.parametrize("nt,npf", GRIDS)
@pytest.mark.parametrize("flags", FLAGS)
def test_multi_step_matches_one_step(nt, npf, flags):
    """n steps in one call and n calls of one-step launches from the same
    state: the cell update differs in FMA contraction at most, so fields agree
    within FP32 rounding of the increments, masks and history alike."""
    steps = 21                          # several launches, rebases inside them, a remainder
    p = _params(flags)
    h, g = _fields(nt, npf, 3)
    many, one = DrainageContext(p, nt, npf, 5e-7), DrainageContext(p, nt, npf, 5e-7)
    one.set_steps_per_launch(1)
    for c in (many, one):
        c.set_fields(h, g)
    dt = 0.3 * one.stats().dt_cfl
    for rep in range(2):                # the second round starts from virtual pole rows
        many.step(steps, dt)
        for _ in range(steps):
            one.step(1, dt)
    hm, gm = many.fields()
    ho, go = one.fields()
    inc = np.abs(ho - h).max()
    assert np.abs(hm - ho).max() <= 2e-5 * inc + 1e-7 * np.float32(5e-7), np.abs(hm - ho).max() / inc
    assert np.abs(gm - go).max() <= 2e-5 * max(np.abs(go - g).max(), 1e-2)
    assert np.array_equal(many.rupture_mask(), one.rupture_mask())
    assert np.array_equal(many.tfe_mask(), one.tfe_mask())
    assert many.current_time() == one.current_time()
    assert many.stats().steps == one.stats().steps
    if flags & DIAG:
        (ma, ca), (mb, cb) = many.history(100), one.history(100)
        assert len(ma) == len(mb) == 2 * steps
        # the volume is linear in h, the limit at most quadratic: the bound on h carries over
        tol = 1e-9 + 2e-5 * inc / h.mean()
        assert np.allclose(ma, mb, rtol=tol, atol=0.0) and np.allclose(ca, cb, rtol=2 * tol, atol=0.0)


@pytest.mark.parametrize("nt,npf,flags,rebase", [
    (128, 256, TFE, 8), (65, 131, TFE | SURF | DIAG, 3), (128, 256, SURF | COPY, 1), (40, 90, MARA | SURF | AVG, 5)])
def test_multi_step_matches_oracle(oracle, nt, npf, flags, rebase):
    p = _params(flags, rebase)
    h, g = _fields(nt, npf, 5)
    ctx = DrainageContext(p, nt, npf, 5e-7)
    ctx.set_fields(h, g)
    dt = 0.3 * ctx.stats().dt_cfl
    q = oracle.Params()
    for name, _ in oracle.Params._fields_:
        setattr(q, name, getattr(p, name))
    sim = oracle.Sim(q, nt, npf)
    sim.set_fields(h, g)
    for _ in range(40):
        sim.step(dt)
    ctx.step(40, dt)
    hc, gc = ctx.fields()
    ho, go = sim.fields()
    inc = np.linalg.norm(hc - ho) / np.linalg.norm(ho - h)
    print("increment rel-L2", inc)
    assert inc <= 1e-5
    assert np.linalg.norm(gc - go) <= 1e-5 * np.linalg.norm(go)


@pytest.mark.parametrize("nt,npf,flags,rebase", [
    (96, 200, TFE | SURF, 8), (3, 7, TFE | SURF | DIAG, 8), (4, 8, TFE, 3), (12, 1024, MARA | SURF | AVG | DIAG, 8),
    (129, 255, MARA | SURF | AVG | DIAG, 5), (128, 256, TFE | DIAG, 8), (300, 601, TFE | SURF | COPY | DIAG, 8),
    (514, 1024, TFE | SURF | DIAG, 8), (1500, 1024, TFE | SURF, 8), (4000, 256, TFE | DIAG, 8)])
def test_multi_step_call_patterns(nt, npf, flags, rebase):
    """Steps in any grouping give the same bits, history included: launches of
    1 .. 8 steps, reads that write the pole rows out between them, and steps
    that are rendered one by one."""
    p = _params(flags, rebase)
    h, g = _fields(nt, npf, 9)
    cam = L.Camera()
    for k, x in enumerate(W.camera(p.bubble_radius)):
        cam.position[k] = x
    cmf = W.spectral_cmf(2).astype(np.float32)
    ref = None
    for groups in ([30], [1] * 30, [2, 3, 4, 5, 6, 7, 3], [8, 1, 8, 1, 8, 4], [29, 1], "rendered"):
        ctx = DrainageContext(p, nt, npf, 5e-7)
        ctx.set_fields(h, g)
        dt = 0.3 * ctx.stats().dt_cfl
        if groups == "rendered":
            L.check(L.lib().sf_drainage_step_spectral(ctx.handle, 17, dt, C.byref(cam), 1.33, L.fptr(cmf)))
            ctx.step(13, dt)
        else:
            for n in groups:
                ctx.step(n, dt)
                ctx.get_thickness(0.0, 0.0)
        out = [*ctx.fields(), *ctx.history(30)]
        if ref is None:
            ref = out
        assert all(np.array_equal(x, y) for x, y in zip(out, ref)), groups
