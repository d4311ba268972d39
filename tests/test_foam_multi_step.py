"""Several steps per launch of small foams (foam_multi_kernel) against the
one-step kernels, over grids at the edges of its rule, and against itself cut
into other launches.

Both run the same cell arithmetic; only the pole means differ, FP64 ring sums
against float-float ones (2^-44 of h a step at 1024 columns), and through
them the roundings of the low word (2^-48 of h): over 40 steps 2^-38 of h.
Surfactant has no ring means: its values are the same bits but for cells that
the thickness decides (none ruptures here)."""
import numpy as np
import pytest

from soap_bubble_simulation_amd.foam import FoamBubble, FoamDrainage, foam_params

pytestmark = pytest.mark.gpu

FOAMS = {
    "smallest": [(3, 2), (4, 8), (3, 10)],
    "one": [(64, 128)],
    "odd": [(17, 34), (40, 78), (63, 126), (5, 1002)],
    "widest": [(12, 1024), (30, 1022)],
    "tall": [(900, 24), (1200, 30)],
    "two_blocks_per_cu": [(18 + k % 20, 36 + 2 * (k % 20)) for k in range(200)],
    "streaming": [(64, 1026), (16, 32)],
}


def _foam(grids, seed=1, rel=0.1):
    rng = np.random.default_rng(seed)
    bub = [FoamBubble(n_theta=a, n_phi=b, bubble_radius=float(rng.uniform(5e-3, 2e-2)),
                      viscosity=float(rng.uniform(1e-3, 4e-3)), h0=5e-7) for a, b in grids]
    fm = FoamDrainage(foam_params(), bub)
    n = fm.length
    fm.set_fields(5e-7 * (1.0 + rel * rng.uniform(-1, 1, n)), 0.5 + 0.2 * rng.uniform(-1, 1, n))
    return fm


@pytest.mark.parametrize("name", list(FOAMS))
def test_matches_one_step_launches(name):
    multi, one = _foam(FOAMS[name]), _foam(FOAMS[name])
    one.set_steps_per_launch(1)
    for steps in (1, 2, 9, 28):
        multi.step(steps)
        one.step(steps)
        (ha, ga), (hb, gb) = multi.fields(), one.fields()
        assert np.all(np.abs(ha - hb) <= 2.0 ** -38 * np.abs(hb)), (name, steps)
        assert np.array_equal(ga, gb), (name, steps)


@pytest.mark.parametrize("name", ["smallest", "odd", "widest", "tall", "two_blocks_per_cu"])
def test_cut_into_other_launches(name):
    a, b = _foam(FOAMS[name]), _foam(FOAMS[name])
    a.step(40)
    for steps in (1, 7, 2, 13, 17):
        b.step(steps)
    assert all(np.array_equal(x, y) for x, y in zip(a.fields(), b.fields()))


def test_held_bubbles_and_explicit_shapes():
    grids = FOAMS["odd"]
    multi, one = _foam(grids), _foam(grids)
    one.set_tile_shapes([9, 9, 9, 9])
    for fm in (multi, one):
        fm.step(3)
        fm.set_active(np.array([1, 0, 1, 0], bool))
        fm.step(21)
        fm.set_active(None)
        fm.step(10)
    (ha, ga), (hb, gb) = multi.fields(), one.fields()
    assert np.all(np.abs(ha - hb) <= 2.0 ** -38 * np.abs(hb)) and np.array_equal(ga, gb)
    held = _foam(grids)
    before = held.split(held.fields()[0])[1]
    held.set_active(np.array([1, 0, 1, 0], bool))
    held.step(19)
    assert np.array_equal(held.split(held.fields()[0])[1][1:-1], before[1:-1])


@pytest.mark.parametrize("launch", ["default", 1, 2])
def test_readers_leave_the_run_alone(launch):
    """Fields and statistics read between steps: the same bits as one run."""
    a, b = _foam(FOAMS["odd"][1:]), _foam(FOAMS["odd"][1:])
    if launch != "default":
        a.set_steps_per_launch(launch)
        b.set_steps_per_launch(launch)
    a.step(33)
    for steps in (1, 5, 8, 3, 16):
        b.step(steps)
        first = b.fields()
        b.stats()
        assert all(np.array_equal(x, y) for x, y in zip(first, b.fields()))
    assert all(np.array_equal(x, y) for x, y in zip(a.fields(), b.fields()))


@pytest.mark.parametrize("name,grids,every", [
    ("more blocks than the rule takes", [(18 + k % 30, 36 + 2 * (k % 30)) for k in range(700)], 40),
    ("one long row", [(40, 1026)] + [(12 + k, 1024 - 2 * k) for k in range(8)], 3),
    ("small", FOAMS["odd"], 2),
    ("two blocks per CU", FOAMS["two_blocks_per_cu"], 40),
])
def test_results_do_not_depend_on_the_active_set(name, grids, every):
    """A few bubbles stepped alone and with their whole foam: the same bits,
    whichever kernels the foam takes.  The films are smooth (1e-4), so that
    the last bits of a pole's mean reach its ring."""
    whole, some = _foam(grids, rel=1e-4), _foam(grids, rel=1e-4)
    mask = np.zeros(len(grids), bool)
    mask[1::every] = True
    some.set_active(mask)
    whole.step(100)
    some.step(100)
    for a, b in zip(whole.fields(), some.fields()):
        for k in np.flatnonzero(mask):
            assert np.array_equal(whole.split(a)[k], some.split(b)[k]), (name, k)


def test_kept_surfactant_waits_for_queued_steps():
    """set_fields that keeps Γ right after queued steps: Γ as they leave it."""
    grids = [(200 + 8 * k, 400 + 16 * k) for k in range(24)]
    a, b = _foam(grids), _foam(grids)
    h = np.full(a.length, 4e-7)
    a.step(200)
    a.set_fields(h)
    b.step(200)
    b.synchronize()
    b.set_fields(h)
    assert np.array_equal(a.fields()[1], b.fields()[1]) and np.array_equal(a.fields()[0], b.fields()[0])
