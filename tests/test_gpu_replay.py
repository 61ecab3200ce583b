"""Replayed chunks.  When a list rebuild inside a chunk overflows its rows,
the step loop restores the chunk's starting state and runs it again with
grown rows; every piece of state that the steps advance (particles, the
Nose-Hoover chain, the thermostat sums, the turn) must come back, so the
trajectory equals a run whose rows never overflowed, bit for bit."""
import sys

import numpy as np
import pytest

from md_engine_amd import systems

pytestmark = pytest.mark.gpu

G = dict(mO=15.9994, mH=1.008, dOH=0.9572, dHH=1.5139, gamma=0.73612446364836)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def water(make, nmol, seed, nh):
    import oracle
    from md_engine_amd import PAIR, PPPM

    box = systems.tip4p2005_box(nmol, seed=seed, min_sep=1.8)
    v = systems.maxwell_boltzmann(box["mass"], 298.0, seed=seed + 1, boltz=systems.REAL_BOLTZ,
                                  mvv_to_eng=systems.REAL_MVV_TO_ENG)
    for o, h1, h2, m in box["mol"]:
        v[o], v[h1], v[h2] = oracle.rattle_one(box["x"][o], box["x"][h1], box["x"][h2], v[o], v[h1], v[h2],
                                               G["mO"], G["mH"])
    e = make()
    inv = np.where(box["mass"] > 0, 1.0 / np.maximum(box["mass"], 1e-30), 0.0)
    e.set_system(box["x"], box["lo"], box["L"], v=v, inv_mass=inv, q=box["q"], types=box["type"])
    e.exclusions_from_bonds(systems.water_bonds(box["mol"]))
    rc = 7.0
    e.nlist_config(rc + 1.0, 1.0)
    eps24, sig6 = systems.water_lj_tables()
    e.lj_set(np.full((3, 3), rc * rc), eps24, sig6)
    e.pppm_set((32, 32, 32), 5, rc, systems.REAL_QQR_TO_ENG)
    e.ewald_real_set(True, -1.0, systems.REAL_QQR_TO_ENG, rc)
    e.rigid_set(box["mol"], G["mO"], G["mH"], G["dOH"], G["dHH"], G["gamma"])
    e.integrator_set(2.0, systems.REAL_FTM_TO_V)
    if nh:
        e.nose_hoover(True, 298.0, 20.0, 10, systems.REAL_BOLTZ, systems.REAL_MVV_TO_ENG)
    return e, PAIR | PPPM


def tight_rows(e, flags):
    """Rows exactly as long as the starting list's longest: a later rebuild
    in which any row grew overflows them and its chunk is replayed."""
    e.compute(flags)
    counts, _ = e.nlist_get()
    cap = max(16, int(counts.max()))
    e.option("row_cap", cap)
    return cap


@pytest.mark.parametrize("graph,trigger", [(0, "forced"), (0, "rows"), (1, "forced"), (1, "rows")])
def test_overflow_replay_with_nose_hoover_is_exact(gpu_engine_factory, graph, trigger):
    """A replayed chunk that starts with a list carried in from an earlier
    build: the replay builds that list again from the positions and box of
    its build, so the rows (and the FP32 summation order they set) are the
    same, and the Nose-Hoover chain and thermostat sums come back with the
    particles.  "forced" replays the third chunk (turns 128-191) through the
    replay_chunk option; "rows" makes the rows exactly as long as the
    starting list's longest, so a later rebuild overflows them."""
    say(f"overflow replay with Nose-Hoover, graph={graph}, trigger={trigger}")
    steps = 384
    ref, flags = water(gpu_engine_factory, 343, 31, nh=True)
    tst, _ = water(gpu_engine_factory, 343, 31, nh=True)
    for e in (ref, tst):
        e.option("graph", graph)
    if trigger == "rows":
        # both engines take the same set-up path and differ only in row length
        cap0 = tight_rows(tst, flags)
        ref.compute(flags)
        ref.option("row_cap", 2 * cap0)
    else:
        tst.option("replay_chunk", 3)
    ref.run(steps, flags)
    tst.run(steps, flags)
    if trigger == "rows":
        cap1 = tst.nlist_stats()["row_cap"]
        say(f"row capacity {cap0} -> {cap1}")
        assert cap1 > cap0, "no rebuild overflowed the tight rows: the replay was not exercised"
    xr, vr = ref.get_system()
    xt, vt = tst.get_system()
    sr, stt = ref.nose_hoover_state(10), tst.nose_hoover_state(10)
    er, et = ref.nose_hoover_energy(), tst.nose_hoover_energy()
    nr, nt = ref.nlist_stats()["rebuilds"], tst.nlist_stats()["rebuilds"]
    ref.close()
    tst.close()
    say(f"  max |dx| {np.abs(xr - xt).max():.2e}, rebuilds {nr} / {nt}")
    assert nr == nt
    assert np.array_equal(xr, xt)
    assert np.array_equal(vr, vt)
    assert np.array_equal(sr, stt)
    assert er == et


@pytest.mark.parametrize("trigger", ["rows", "forced"])
def test_batch_replay_keeps_replicas_in_step(gpu_engine_factory, trigger):
    """Three replicas in one batch, one with tight rows (or made to replay
    its second chunk): its replay replays the chunk for every replica, and
    each still equals its own single run."""
    from md_engine_amd._lib import run_batch

    say(f"batch replay ({trigger})")
    steps = 128
    seeds = (41, 42, 43)
    singles = []
    for s in seeds:
        e, flags = water(gpu_engine_factory, 216, s, nh=False)
        e.option("graph", 1)
        e.run(steps, flags)
        singles.append(e.get_system())
        e.close()
    batch = []
    for s in seeds:
        e, flags = water(gpu_engine_factory, 216, s, nh=False)
        batch.append(e)
    if trigger == "rows":
        cap0 = tight_rows(batch[1], flags)
    else:
        batch[1].option("replay_chunk", 2)
    run_batch(batch, steps, flags)
    if trigger == "rows":
        cap1 = batch[1].nlist_stats()["row_cap"]
        say(f"replica 1 row capacity {cap0} -> {cap1}")
        assert cap1 > cap0
    for e, (xs, vs) in zip(batch, singles):
        xb, vb = e.get_system()
        assert np.array_equal(xb, xs)
        assert np.array_equal(vb, vs)
    for e in batch:
        e.close()


@pytest.mark.parametrize("graph", [0, 1])
def test_replay_under_a_barostat_is_exact(gpu_engine_factory, graph):
    """The barostat dilates the sites after a step's forces, and the next
    step's first kick takes those forces: a chunk replayed from a carried list
    takes them too, not the forces at the dilated positions."""
    say(f"replay under a barostat, graph={graph}")
    out = []
    for chunk in (0, 2):
        e, flags = water(gpu_engine_factory, 343, 33, nh=False)
        e.thermostat(True, 298.0, 10, 0.0, systems.REAL_BOLTZ, systems.REAL_MVV_TO_ENG)
        e.barostat(True, 1.0, 100.0, 1, 10.0, 1e-5, mvv_to_eng=systems.REAL_MVV_TO_ENG)
        e.option("graph", graph)
        e.option("replay_chunk", chunk)
        e.run(192, flags)
        x, v = e.get_system()
        out.append((x, v, e.get_box()[1], e.nlist_stats()["rebuilds"]))
        e.close()
    (xr, vr, Lr, nr), (xt, vt, Lt, nt) = out
    say(f"  max |dx| {np.abs(xr - xt).max():.2e}, rebuilds {nr} / {nt}")
    assert nr == nt
    assert np.array_equal(Lr, Lt)
    assert np.array_equal(xr, xt)
    assert np.array_equal(vr, vt)


def shrinking_water(make, e3b=False):
    """A box that loses a cell per axis near step 50 of a run: every step
    shrinks it by the largest dilation."""
    box = systems.tip4p2005_box(283, seed=35, min_sep=1.8)
    import oracle
    from test_gpu_water_md import start_velocities, water_md_engine

    e, flags = water_md_engine(make, box, start_velocities(oracle, box, seed=8), rc=7.0, skin=1.0, sz=(32, 32, 32),
                               order=5, e3b=e3b, dt=1.0)
    e.thermostat(True, 298.0, 5, 0.0, systems.REAL_BOLTZ, systems.REAL_MVV_TO_ENG)
    e.barostat(True, 1e9, 1.0, 1, bulk_modulus=1e-3, max_dilation=4e-4, mvv_to_eng=systems.REAL_MVV_TO_ENG)
    return e, flags, box


def test_replay_of_a_chunk_with_a_grid_change(gpu_engine_factory):
    """Eager steps under a barostat set a coarser cell grid up inside a chunk;
    replayed from a carried list, the chunk starts on its own grid again, with
    the sites in that grid's order, and changes it at the same step."""
    say("replay of a chunk with a grid change")
    out = []
    for chunk in (0, 1):
        e, flags, _ = shrinking_water(gpu_engine_factory)
        e.option("graph", 0)
        e.run(8, flags)
        cells = e.nlist_stats()["cells"]
        e.option("replay_chunk", chunk)
        e.run(64, flags)
        st = e.nlist_stats()
        say(f"  cells {cells} -> {st['cells']}, rebuilds {st['rebuilds']}")
        assert tuple(cells) == (5, 5, 10) and tuple(st["cells"]) == (4, 4, 9)
        out.append((*e.get_system(), e.get_box()[1], st["rebuilds"]))
        e.close()
    assert out[0][3] == out[1][3]
    for a, b in zip(out[0][:3], out[1][:3]):
        assert np.array_equal(a, b)


def test_overflow_before_a_grid_change_is_replayed(gpu_engine_factory):
    """A rebuild overflows its rows, and later in the same chunk the box loses
    a cell: the build on the new grid makes room by itself, and the chunk is
    replayed all the same, on the grid it started with."""
    say("row overflow before a grid change in one chunk")
    out = []
    for scale in (2, 1):
        e, flags, box = shrinking_water(gpu_engine_factory)
        e.option("graph", 0)
        cap = tight_rows(e, flags)
        e.option("row_cap", scale * cap)
        cells = [e.nlist_stats()["cells"]]
        e.run(64, flags)
        st = e.nlist_stats()
        cells.append(st["cells"])
        say(f"  rows {scale * cap} -> {st['row_cap']}, cells {cells}, rebuilds {st['rebuilds']}")
        assert tuple(cells[1]) != tuple(cells[0])
        out.append((*e.get_system(), e.get_box()[1], st["rebuilds"]))
        e.close()
    assert out[0][3] == out[1][3]
    for a, b in zip(out[0][:3], out[1][:3]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("ensemble", ["rescale", "nose", "npt"])
@pytest.mark.parametrize("graph", [0, 1])
def test_overflow_of_molecule_rows_is_exact(gpu_engine_factory, graph, ensemble):
    """E3B molecule rows exactly as long as the starting list's longest: a
    rebuild somewhere in a chunk overflows them, also where the chunk's last
    rebuild fits again, and the replayed chunks equal those of loose rows."""
    import oracle
    from test_gpu_water_md import start_velocities, water_md_engine

    say(f"overflow of E3B molecule rows, graph={graph}, {ensemble}")
    box = systems.tip4p2005_box(441, seed=37, min_sep=1.8)
    v = start_velocities(oracle, box, seed=8)
    kb, mvv = systems.REAL_BOLTZ, systems.REAL_MVV_TO_ENG

    def longest(e):
        L = e.get_box()[1]
        o = e.get_system()[0][box["mol"][:, 0]]
        d = o[:, None] - o[None]
        d -= L * np.rint(d / L)
        return int(((d ** 2).sum(-1) < 7.2 ** 2).sum(1).max() - 1)

    out, grown = [], 0
    for kind in ("loose", "tight", "sampled"):
        e, flags = water_md_engine(gpu_engine_factory, box, v, rc=7.0, skin=1.0, sz=(32, 32, 32), order=5, e3b=True,
                                   dt=2.0)
        if ensemble == "nose":
            e.nose_hoover(True, 298.0, 100.0, 10, kb, mvv)
        else:
            e.thermostat(True, 298.0, 10, 0.0, kb, mvv)
        if ensemble == "npt":
            e.barostat(True, 1.0, 1000.0, 1, mvv_to_eng=mvv)
        e.option("graph", graph)
        e.run(16, flags)
        most = longest(e)
        # the next run's first build finds this longest row
        e.option("e3b_row_cap", most if kind == "tight" else 2 * most)
        if kind == "sampled":
            for _ in range(48):
                e.run(4, flags)
                grown = max(grown, longest(e))
        else:
            for _ in range(3):
                e.run(64, flags)
            out.append((*e.get_system(), e.get_box()[1], e.nlist_stats()["rebuilds"]))
        e.close()
    say(f"  longest row {most} at the start, {grown} later")
    assert grown > most, "no row grew past the tight capacity"
    assert out[0][3] == out[1][3]
    for a, b in zip(out[0][:3], out[1][:3]):
        assert np.array_equal(a, b)


def test_replay_after_the_barostat_was_switched_off(gpu_engine_factory):
    """The forces carried into a constant-volume run are still those before
    the barostat's last dilation."""
    say("replay after the barostat was switched off")
    out = []
    for chunk in (0, 1):
        e, flags = water(gpu_engine_factory, 343, 33, nh=False)
        e.barostat(True, 1.0, 100.0, 1, 10.0, 1e-4, mvv_to_eng=systems.REAL_MVV_TO_ENG)
        e.run(20, flags)
        e.barostat(False)
        e.option("replay_chunk", chunk)
        e.run(40, flags)
        out.append(e.get_system())
        e.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_replay_with_a_long_range_interval(gpu_engine_factory):
    """Between the steps that evaluate the mesh its stored forces are added:
    a chunk entered in between is replayed from the forces it was entered with."""
    say("replay with a long-range interval")
    out = []
    for chunk in (0, 1):
        e, flags = water(gpu_engine_factory, 343, 33, nh=False)
        e.pppm_interval(3)
        e.run(20, flags)
        e.option("replay_chunk", chunk)
        e.run(40, flags)
        out.append(e.get_system())
        e.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
