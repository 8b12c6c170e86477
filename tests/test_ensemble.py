"""Batched ensembles (mercurydpm_fork_amd/ensemble.py): independent heaps laid
side by side in one engine context run exactly as they run alone, because
no interaction range reaches across the gap between their tiles."""
import numpy as np
import pytest

import oracle_lib
from mercurydpm_fork_amd import dem, ensemble as E, scenarios as S


def members(sizes, seed=3):
    sp = E.calibration_species()
    return [E.heap(n, seed + k, sp) for k, n in enumerate(sizes)]


def test_pack_layout_and_checks():
    ms = members([50, 300, 120, 800, 20])
    p = E.pack(ms)
    st = p.scenario.state
    assert st.n == sum(m.state.n for m in ms)
    assert len(np.unique(st.id)) == st.n
    # the tiles are apart by at least the gap, so no two members can touch
    for a in range(len(ms)):
        for b in range(a + 1, len(ms)):
            xa, xb = p.member(a, st.x) + p.offsets[a], p.member(b, st.x) + p.offsets[b]
            lo_a, hi_a = xa[:, :2].min(0), xa[:, :2].max(0)
            lo_b, hi_b = xb[:, :2].min(0), xb[:, :2].max(0)
            sep = np.maximum(lo_b - hi_a, lo_a - hi_b).max()
            assert sep >= p.gap
    for k, m in enumerate(ms):  # shifting there and back rounds in the last bit
        np.testing.assert_allclose(p.member(k, st.x), m.state.x, rtol=0, atol=1e-12)
    assert p.check_separated(st.x)
    bad = members([30])[0]
    bad.periodic = [S.periodic_boundary(0, 0.0, 5.0)]
    with pytest.raises(ValueError):
        E.pack([ms[0], bad])


def _run(sc, steps, engine):
    e = engine()
    S.apply(e, sc)
    e.compute_forces()
    e.step(steps)
    return e


def test_ensemble_equals_members_on_oracle():
    """On the oracle: three heaps packed, 150 steps, each member's positions
    equal its own run's to round-off (the packed run sums a particle's
    forces in another order only through the ghost-free pair loop)."""
    ms = members([60, 150, 90])
    p = E.pack(ms)
    x = _run(p.scenario, 150, oracle_lib.engine).download()["x"]
    assert p.check_separated(x)
    for k, m in enumerate(ms):
        xk = _run(m, 150, oracle_lib.engine).download()["x"]
        np.testing.assert_allclose(p.member(k, x), xk, rtol=0, atol=1e-10)


@pytest.mark.gpu
def test_ensemble_equals_members_on_engine():
    """On the engine: six heaps of 100 to 1500 spheres packed, 400 steps:
    every member's contacts (ids mapped back) and positions equal its own
    engine run's (positions to round-off of differently ordered force sums)."""
    sizes = [100, 1500, 300, 800, 150, 600]
    ms = members(sizes, seed=11)
    p = E.pack(ms)
    g = _run(p.scenario, 400, dem.Engine)
    x = g.download()["x"]
    assert p.check_separated(x)
    cp = g.contacts()
    for k, m in enumerate(ms):
        e = _run(m, 400, dem.Engine)
        np.testing.assert_allclose(p.member(k, x), e.download()["x"], rtol=0, atol=1e-9)
        lo, hi = p.first[k], p.first[k + 1]
        own = {(int(a) - lo, int(b) if b & dem.DEM_WALL_KEY else int(b) - lo)
               for a, b in zip(cp.p_id, cp.i_id) if lo <= a < hi}
        assert own == e.contacts().keys()


# ---------------------------------------------------------------------------
# Calibration heaps with per-simulation parameters and walls
# (Drivers/Calibration/CalibrationHeap.cpp)
# ---------------------------------------------------------------------------

def heap_members(sizes, seed=5):
    rng = np.random.default_rng(seed)
    ps = [E.HeapParams(int(n), float(rng.uniform(0.1, 0.8)), float(rng.uniform(0.0, 0.1)),
                       float(rng.uniform(0.5, 0.95)), int(seed * 1000 + k)) for k, n in enumerate(sizes)]
    return [E.calibration_heap(p) for p in ps]


def test_heap_packing_and_wall_groups():
    """Each heap: spheres inside its casing, above its base, not overlapping;
    the packed scenario gives heap k species 2k (casing 2k + 1), walls 2k and
    2k + 1 at its centre, and the wall group (2k, 2) to its particles."""
    ms = heap_members([120, 300, 80])
    for sc in ms:
        x, r, R = sc.state.x, sc.state.radius, sc.info["base_radius"]
        d = np.sqrt(((x[:, None] - x[None]) ** 2).sum(-1))
        np.fill_diagonal(d, np.inf)
        assert np.all(d >= r[:, None] + r[None] - 1e-12)
        assert np.all(np.hypot(x[:, 0], x[:, 1]) + r <= R + 1e-12) and np.all(x[:, 2] >= r - 1e-12)
    for schedule in ("grid", "shelf"):
        ens = E.pack_heaps(ms, schedule=schedule)
        sc = ens.scenario
        first, count = sc.wall_groups
        assert list(first) == [0, 0, 2, 2, 4, 4] and list(count) == [2, 0, 2, 0, 2, 0]
        for k in range(3):
            lo, hi = ens.id_first[k], ens.id_first[k + 1]
            assert np.all(sc.state.species[lo:hi] == 2 * k)
            for w in (sc.walls[2 * k], sc.walls[2 * k + 1]):
                assert (w.position[0], w.position[1]) == (ens.offsets[k, 0], ens.offsets[k, 1])
            assert sc.walls[2 * k].species == 2 * k and sc.walls[2 * k + 1].species == 2 * k + 1
        # bases at least the gap apart
        for a in range(3):
            for b in range(a + 1, 3):
                gap = np.hypot(*(ens.offsets[a, :2] - ens.offsets[b, :2])) - ens.base_radius[a] - ens.base_radius[b]
                assert gap >= 8.0 * 0.6 - 1e-9
        # the table: each heap's own 2 x 2 block
        ns = 6
        for k in range(3):
            own = S.species_table(ms[k].species)
            for a in range(2):
                for b in range(2):
                    assert bytes(sc.table()[(2 * k + a) * ns + 2 * k + b]) == bytes(own[2 * a + b])


def _heap_run(sc, steps, engine, lift_at=None, first_count=None):
    """steps steps; at lift_at, the casing goes (alone: removeLastObject;
    packed: the given wall groups)."""
    e = engine()
    S.apply(e, sc)
    e.compute_forces()
    if lift_at is None:
        e.step(steps)
        return e
    e.step(lift_at)
    if first_count is None:
        e.set_walls(sc.walls[:1])
    else:
        e.set_wall_groups(*first_count)
    e.step(steps - lift_at)
    return e


def _lifted(ens, which):
    first, count = (np.array(a) for a in ens.scenario.wall_groups)
    count[2 * np.asarray(which)] = 1
    return first, count


def test_heap_members_on_oracle():
    """On the oracle: three heaps with their own parameters packed (wall
    groups), 2500 steps (the fill falls about 3 diameters), the first heap's
    casing lifted at step 1500: every heap's positions equal its own run's
    (alone, WallHandler::removeLastObject at the same step) to round-off
    (the tile offset rounds every position, and 2500 steps of collisions
    amplify it to a few 1e-10)."""
    ms = heap_members([150, 260, 200], seed=7)
    ens = E.pack_heaps(ms)
    e = _heap_run(ens.scenario, 2500, oracle_lib.engine, 1500, _lifted(ens, [0]))
    x = e.download()["x"]
    assert any(b & dem.DEM_WALL_KEY for b in e.contacts().i_id)
    for k, m in enumerate(ms):
        xk = _heap_run(m, 2500, oracle_lib.engine, 1500 if k == 0 else None).download()["x"]
        lo, hi = ens.id_first[k], ens.id_first[k + 1]
        np.testing.assert_allclose(x[lo:hi] - ens.offsets[k], xk, rtol=0, atol=1e-8)


@pytest.mark.gpu
def test_heap_members_engine_vs_oracle():
    """On the engine: four heaps of 300 to 1500 spheres with their own
    sliding/rolling friction and restitution packed with wall groups, 2000
    steps, casings of heaps 1 and 3 lifted at step 1000: each heap's contacts
    (ids mapped back) equal those of its own run on the oracle, positions to
    round-off of differently ordered force sums and of the tile offset,
    amplified by 2000 steps of dense collisions (measured up to 1e-8)."""
    ms = heap_members([300, 1500, 700, 450], seed=9)
    ens = E.pack_heaps(ms)
    g = _heap_run(ens.scenario, 2000, dem.Engine, 1000, _lifted(ens, [1, 3]))
    x = g.download()["x"]
    cp = g.contacts()
    for k, m in enumerate(ms):
        o = _heap_run(m, 2000, oracle_lib.engine, 1000 if k in (1, 3) else None)
        lo, hi = ens.id_first[k], ens.id_first[k + 1]
        np.testing.assert_allclose(x[lo:hi] - ens.offsets[k], o.download()["x"], rtol=0, atol=1e-7)
        own = {(int(a) - lo, int(b) - 2 * k if b & dem.DEM_WALL_KEY else int(b) - lo)
               for a, b in zip(cp.p_id, cp.i_id) if lo <= a < hi}
        want = o.contacts().keys()
        assert own == want, (k, len(own ^ want))
        assert any(b & dem.DEM_WALL_KEY for _, b in want)


@pytest.mark.gpu
def test_heap_protocol_runs_to_angles_of_repose():
    """The CalibrationHeap protocol on six packed heaps (500 to 2000 spheres)
    for 30,000 steps: every casing is lifted once its heap has settled,
    spheres that fall off the base are deleted, and the angles of repose of
    the heaps (after twice the fill time once settled, else at the end) lie
    between 5 and 60 degrees."""
    ps = E.draw_heap_params(6, 3, n_range=(500, 2000))
    ens = E.pack_heaps([E.calibration_heap(p) for p in ps])
    g = dem.Engine()
    S.apply(g, ens.scenario)
    g.compute_forces()
    run = E.run_heap_protocol(g, ens, 30000)
    assert np.all(np.isfinite(run.fill_time)), run.fill_time
    assert run.removed > 0
    assert np.all((run.angle_at_end > 5) & (run.angle_at_end < 60)), run.angle_at_end
    ok = np.isfinite(run.angle_of_repose)
    assert ok.sum() >= 1, run.angle_of_repose
    assert np.all((run.angle_of_repose[ok] > 5) & (run.angle_of_repose[ok] < 60)), run.angle_of_repose


@pytest.mark.gpu
def test_autotune_picks_the_fastest_candidate():
    """The autotuner times every (layout, skin) candidate from the same
    warmed-up state and returns the fastest; a skin whose lists would
    overflow is left out rather than failing the search."""
    params = E.draw_heap_params(6, 11, n_range=(500, 1500))
    members = [E.calibration_heap(p) for p in params]
    sch, skin, table = E.autotune(members, skins=(0.2, 0.8, 2.4), steps=50, warm_steps=500)
    assert {row["schedule"] for row in table} == {"shelf", "grid"}
    best = min(table, key=lambda row: row["ms_per_step"])
    assert (sch, skin) == (best["schedule"], best["skin"])
    # the picked set-up runs the protocol
    ens = E.pack_heaps(members, schedule=sch)
    e = dem.Engine(skin=skin)
    S.apply(e, ens.scenario)
    e.compute_forces()
    run = E.run_heap_protocol(e, ens, 2000)
    e.close()
    assert run.steps == 2000 and set(run.seconds) == {"step", "check", "delete"}


def test_deletion_sequence_is_the_scan():
    """deletion_sequence against the reference's scan written out
    (DeletionBoundary.cc:197-219 with ParticleHandler::removeObject), over
    every subset of up to 8 particles and random ones of 60."""
    def scan(n, doomed):
        order, dead, seq, i = np.arange(n), np.zeros(n, bool), [], 0
        dead[doomed] = True
        while i < n:
            if dead[i]:
                seq.append(i)
                dead[i], order[i] = dead[n - 1], order[n - 1]
                n -= 1
            else:
                i += 1
        return np.array(seq, np.int64), order[:n]

    cases = [(n, [k for k in range(n) if m >> k & 1]) for n in range(9) for m in range(1 << n)]
    rng = np.random.default_rng(1)
    cases += [(60, rng.permutation(60)[:rng.integers(0, 61)]) for _ in range(300)]
    for n, doomed in cases:
        for got, want in zip(E.deletion_sequence(n, doomed), scan(n, np.asarray(doomed, np.int64))):
            np.testing.assert_array_equal(got, want)
