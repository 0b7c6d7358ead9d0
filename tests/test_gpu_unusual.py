"""Colour passes on states outside the single-precision filter's bounds
(kf_device.hpp, F32Filter): their decisions are the exact arithmetic's,
and every read stays inside the particles' arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pp():
    import patchyparticles_amd as pp
    pp.lib()
    return pp


TAG_TRIAL_A, TAG_SHIFT, TAG_COLOUR = 0, 8, 9


def _cell_coord(x, shift, inv_box, n):
    t = (x - shift) * inv_box
    t = t - np.floor(t)
    i = int(t * float(n)) if t == t else 0
    return min(i, n - 1)


def _free_particle(oracle, p, box, n, sweeps, trials, seed, disp_max):
    """The walk of a single particle: a trial is accepted if it stays in the
    cell of the sweep's grid (cell_coord, FP64).  Returns its end and the
    number of accepted trials."""
    u01 = lambda w: float(w) * 2.0 ** -32
    key = [seed, 0]
    p, inv, accepted = [float(v) for v in p], 1.0 / box, 0
    for sweep in range(sweeps):
        w = oracle.philox([0, TAG_SHIFT, sweep, 0], key)
        shift = [u01(w[k]) * (box / n) for k in range(3)]
        at = [_cell_coord(p[k], shift[k], inv, n) for k in range(3)]
        colour = (at[0] & 1) << 2 | (at[1] & 1) << 1 | at[2] & 1
        ctr = np.array([[(at[0] * n + at[1]) * n + at[2], TAG_TRIAL_A | colour << 8 | t << 16, sweep, 0] for t in range(trials)])
        for w in oracle.philox_n(ctr, np.array([key] * trials)):
            q = [p[k] + (u01(w[1 + k]) - 0.5) * disp_max for k in range(3)]
            if all(_cell_coord(q[k], shift[k], inv, n) == at[k] for k in range(3)):
                p, accepted = q, accepted + 1
    return np.array(p), accepted


@pytest.mark.parametrize("disp_max", [0.3, 1.1])
@pytest.mark.parametrize("at", [3.0, -5e6, 3e7, 1e11, -1e13, 1e14])
def test_in_cell_test_at_large_coordinates(pp, oracle, at, disp_max):
    """One particle at coordinates whose own spacing is up to 1/64: it leaves or
    stays in its cell as FP64 says, trial by trial, in every team width."""
    box, n, sweeps, trials, seed = 8.0, 6, 150, 16, 5
    p = np.array([at, 1.5 + at, 2.25 - at])
    want, accepted = _free_particle(oracle, p, box, n, sweeps, trials, seed, disp_max)
    assert 0.2 * sweeps * trials < accepted < sweeps * trials
    for kw in (dict(threads_per_cell=16, block_size=64), dict(threads_per_cell=32), dict(threads_per_cell=64), dict(launch=3)):
        with pp.System(p[None], np.eye(3)[None], np.full(3, box), T=0.1, seed=seed, disp_max=disp_max, trials_per_cell=trials,
                       **kw) as s:
            assert s.grid()[0] == [n] * 3
            s.do_ensemble(sweeps)
            r, _, _ = s.state()
            assert s.counters()["accepted"][0] == accepted and np.array_equal(r[0], want), kw


COOP, DEPS = 2, 3


@pytest.mark.parametrize("rho,occupancy", [(0.05, 0.0), (0.3, 0.0), (0.3, 6.0)])
@pytest.mark.parametrize("trials", [0, 16])
def test_coordinates_that_are_not_finite(pp, oracle, rho, occupancy, trials):
    """A particle with a NaN or infinite coordinate has no neighbour: its moves
    find no overlap and no bond, and the other particles move as without it in
    reach.  Cells of few and of many neighbours (the occupancies), so that
    teams have empty slots, full ones and neighbours beyond them; every form
    of the passes gives the same trajectory."""
    r, O, box = pp.generate(1500, rho, 21)
    bad = [3, 40, 41, 333, 1499]
    r[bad, [0, 1, 2, 0, 1]] = [np.nan, np.inf, -np.inf, np.nan, np.nan]
    r[333] = np.nan
    fine = np.setdiff1d(np.arange(len(r)), bad)
    got = []
    for kw in (dict(threads_per_cell=32), dict(threads_per_cell=16, block_size=64), dict(threads_per_cell=64),
               dict(launch=COOP), dict(launch=DEPS), dict(copies=2), dict(copies=2, threads_per_cell=16, block_size=64)):
        copies = kw.pop("copies", 1)
        with pp.System.batch([r] * copies, [O] * copies, [box] * copies, [dict(T=0.12)] * copies, seed=9,
                             cell_occupancy=occupancy, trials_per_cell=trials, **kw) as s:
            s.do_ensemble(20)
            bonds, ov, total, any_ov = s.energy(0)
            rr, OO, _ = s.state(0)
            c = s.counters(0)
            assert not any_ov and c["bonds"] == total and not bonds[bad].any(), kw
            ob, oov, ototal = oracle.energy(rr[fine], OO[fine], box)
            assert np.array_equal(bonds[fine], ob) and not oov.any() and ototal == total, kw
            got.append((rr, OO, c["tries"], c["accepted"]))
    assert not np.isfinite(got[0][0][bad]).all(axis=1).any() and np.isfinite(got[0][0][fine]).all()
    for x in got[1:]:
        for a, b in zip(got[0], x):
            assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("disp_max", [0.9, 1.2, 2.5, 6.9, 7.1, 9.3, 40.0])
def test_steps_longer_than_a_cell_and_round_the_box(pp, oracle, disp_max):
    """Steps (up to disp_max / 2 per axis) that leave the cell, and from
    disp_max 6.96 on some that come round the 4-cell box into it: one particle
    walks as FP64 says, and many never overlap and keep their bonds' count, in
    every form of the passes."""
    r, O, box = pp.generate(20, 0.2, 4)
    sweeps, trials, seed = 400, 16, 11
    want, accepted = _free_particle(oracle, r[0], float(box[0]), 4, sweeps, trials, seed, disp_max)
    got = []
    for kw in (dict(threads_per_cell=16, block_size=64), dict(threads_per_cell=32), dict(threads_per_cell=64), dict(launch=COOP),
               dict(launch=DEPS)):
        kw.update(T=0.12, seed=seed, disp_max=disp_max, trials_per_cell=trials)
        with pp.System(r[:1], O[:1], box, **kw) as s:
            assert s.grid()[0] == [4] * 3
            s.do_ensemble(sweeps)
            assert s.counters()["accepted"][0] == accepted and np.array_equal(s.state()[0][0], want), kw
        with pp.System(r, O, box, **kw) as s:
            for _ in range(8):
                s.do_ensemble(sweeps // 8)
                rr, OO, _ = s.state()
                b, ov, total, any_ov = s.energy()
                ob, oov, ototal = oracle.energy(rr, OO, box, brute=True)
                assert not any_ov and not oov.any() and np.array_equal(b, ob), kw
                assert s.counters()["bonds"] == total == ototal, kw
            got.append((rr, OO, s.counters()["accepted"]))
    for x in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], x))


@pytest.mark.parametrize("scale", [1.0, 1.015, 1.3])
@pytest.mark.parametrize("offset", [0, 10 ** 6, 10 ** 9])
def test_orientations_and_coordinates_past_the_bounds(pp, oracle, scale, offset):
    """Particles some boxes away from the first (coordinates to 10^10) and
    matrices whose entries pass 1.01: bonds are the exact arithmetic's, and the
    team widths agree."""
    r, O, _ = pp.generate(600, 0.4, 8)
    box = np.full(3, 11.5)
    r = r * (11.5 / (600 / 0.4) ** (1 / 3))
    rng = np.random.default_rng(3)
    r = r + box * rng.integers(-offset, offset + 1, r.shape)
    O = O * scale
    got = []
    for kw in (dict(threads_per_cell=16, block_size=64), dict(threads_per_cell=32), dict(threads_per_cell=64), dict(launch=DEPS)):
        with pp.System(r, O, box, T=0.12, seed=2, trials_per_cell=8, **kw) as s:
            s.do_ensemble(40)
            rr, OO, _ = s.state()
            b, ov, total, any_ov = s.energy()
            ob, oov, ototal = oracle.energy(rr, OO, box)
            assert not any_ov and not oov.any() and np.array_equal(b, ob), kw
            assert s.counters()["bonds"] == total == ototal > 0, kw
            got.append((rr, OO, s.counters()["accepted"]))
    for x in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], x))


@pytest.mark.parametrize("trials", [0, 8])
@pytest.mark.parametrize("occupancy", [0.0, 6.0])
def test_overlaps_left_by_a_refused_upload(pp, occupancy, trials):
    """A refused upload leaves its particles: the passes then move them apart,
    and a bond that an overlapping pair has at the present position counts
    wherever the pair is found, in a lane's slots or beyond them (occupancy 6:
    more neighbours than any team's slots)."""
    r, O, box = pp.generate(1500, 0.5, 6)
    O[:] = O[0]
    got = []
    for kw in (dict(threads_per_cell=16, block_size=64), dict(threads_per_cell=32), dict(threads_per_cell=64), dict(launch=DEPS)):
        with pp.System(r, O, box, T=0.12, seed=2, cell_occupancy=occupancy, trials_per_cell=trials, kf_cosmax=0.5, **kw) as s:
            with pytest.raises(pp.PPError) as e:
                s.upload(0, r * 0.97, O, box * 0.97)
            assert e.value.status == 3  # PP_ERR_OVERLAP
            s.do_ensemble(30)
            got.append(s.state() + (s.counters()["accepted"],))
    assert got[0][3][0] > 10000
    for x in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], x))
