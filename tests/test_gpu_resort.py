"""The two-launch re-sort (bin_body, sort_body) at the shapes where it can go
wrong, through the neighbor list it leaves: rows against the oracle bit for bit.

* cells that hold far more atoms than the register and LDS paths take (a dense
  cluster in a large box: the walk through the cell's list);
* a grid with fewer cells than one chunk, and one with several rounds per chunk
  (a sparse gas over hundreds of thousands of cell slots);
* exclusion rows longer than a wave's registers;
* steps of free atoms (first half kick, check and refresh fused; captured: the
  decisions in the binning) against the separate launches, bit for bit;
* what a list read back depends on: parts left out, captured builds that did
  not run, a box turned on its side.
"""
import numpy as np
import pytest

from md_engine_amd import PAIR
from test_gpu_parity import assert_same_lists, oracle_rows_by_id

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)


def _list_engine(factory, x, L, rlist, skin, q=None):
    e = factory()
    e.set_system(x, np.zeros(3), L, q=q, inv_mass=np.ones(len(x)))
    e.lj_set([[(rlist - skin) ** 2]], [[24.0]], [[1.0]])
    e.nlist_config(rlist, skin)
    return e


@pytest.mark.parametrize("shape", ["cluster", "one_chunk", "sparse"])
def test_resort_lists_exact(orc, gpu_engine_factory, shape):
    say(f"re-sort, {shape}")
    rng = np.random.default_rng(5)
    if shape == "cluster":
        # 3,000 atoms in one cell (beyond the 2,048 ranked in LDS), 500 around them
        L = np.full(3, 24.0)
        x = np.concatenate([rng.uniform(11.0, 11.2, (3000, 3)), rng.uniform(0, 24, (500, 3))])
        rlist = 2.5
    elif shape == "one_chunk":
        L = np.array([6.1, 6.3, 7.0])
        x = rng.uniform(0, 1, (333, 3)) * L
        rlist = 2.9
    else:
        # 2 x (124 x 124 x 249) cell slots: several rounds of 256 cells per workgroup
        L = np.full(3, 125.0)
        x = rng.uniform(0, 125, (20011, 3))
        rlist = 2.0
    q = np.where(rng.random(len(x)) < 0.4, 0.3, 0.0)
    if shape == "cluster":
        q[:3000] = 0.0  # one cell slot
    e = _list_engine(gpu_engine_factory, x, L, rlist, 0.3, q=q)
    for k in range(2):  # the second build starts from the first one's order
        e.nlist_update(force=True)
        gc, grows = e.nlist_get()
        oc, orows, _ = oracle_rows_by_id(orc, x, np.zeros(3), L, rlist, brute=False)
        assert_same_lists(gc, grows, oc, orows)
        x = x + rng.normal(0, 0.2, x.shape)
        e.set_positions(x)
    e.close()


def test_long_exclusion_rows(orc, gpu_engine_factory):
    """Rows of 3, 70 and 100 exclusions: registers, LDS and beyond one per lane."""
    say("long exclusion rows")
    rng = np.random.default_rng(6)
    n, L = 400, np.full(3, 9.0)
    x = rng.uniform(0, 9, (n, 3))
    e = _list_engine(gpu_engine_factory, x, L, 2.5, 0.3)
    partners = [set() for _ in range(n)]
    for i, m in ((3, 3), (50, 70), (51, 100)):
        for j in rng.choice([k for k in range(100, n)], m, replace=False):
            partners[i].add(int(j))
            partners[int(j)].add(i)
    off = np.concatenate([[0], np.cumsum([len(p) for p in partners])]).astype(np.int32)
    tagged = np.array([j | (1 + j % 3) << 30 for p in partners for j in sorted(p)], np.uint32)
    e.exclusions_set(off, tagged)
    e.nlist_update(force=True)
    gc, grows = e.nlist_get()
    tags = {(i, j): 1 + j % 3 for i in range(n) for j in partners[i]}
    oc, orows, _ = oracle_rows_by_id(orc, x, np.zeros(3), L, 2.5, brute=True)
    for i in range(n):
        want = [int(r) & 0x3FFFFFFF for r in orows[i]]
        assert [int(r) for r in grows[i]] == [j | (tags.get((i, j), 0) << 30) for j in want], i
    e.close()


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("n", [256, 257, 4000])
def test_fused_first_half_equals_separate(orc, gpu_engine_factory, n, graph):
    """Free atoms, eager and captured steps: kick, check and refresh in one
    launch (captured: the decisions in the binning) give the separate
    launches' trajectory bit for bit."""
    say(f"fused first half, {n} atoms, graph {graph}")
    from md_engine_amd import systems

    x, L, lo = systems.fcc_lj(10, 0.8442)
    x = x[:n] if n == 4000 else x[np.random.default_rng(1).choice(4000, n, replace=False)]
    v = systems.maxwell_boltzmann(np.ones(n), 1.2, seed=4)
    out = []
    for fuse in (1, 0):
        e = gpu_engine_factory()
        e.set_system(x, lo, L, v=v, inv_mass=np.ones(n))
        e.lj_set([[6.25]], [[24.0]], [[1.0]])
        e.nlist_config(2.8, 0.3)
        e.integrator_set(0.005, 1.0)
        e.option("fuse_step", fuse)
        e.option("graph", graph)
        e.run(150, PAIR)
        st = e.nlist_stats()
        out.append((*e.get_system(), st["rebuilds"], st["violations"]))
        e.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert out[0][2] == out[1][2] and out[0][2] > 3
    assert out[0][3] == 0


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("team", [0, 16])
def test_whole_list_from_partial_rows(orc, gpu_engine_factory, graph, team):
    """Builds leave out the parts of the rows that no kernel reads (an oxygen's
    charged partners, a charged site's charge-free ones); the list that is read
    back is whole all the same, after runs and after the force terms change to
    ones that read more, and the forces then are those of a fresh engine."""
    say(f"partial rows, graph {graph}, team {team}")
    from md_engine_amd import E3B, PPPM, systems
    from test_gpu_water_md import start_velocities, water_md_engine

    box = systems.tip4p2005_box(343, seed=36, min_sep=1.8)
    n, L = len(box["x"]), box["L"]
    excl = orc.exclusions_bfs(n, systems.water_bonds(box["mol"]))

    def make(v):
        e, flags = water_md_engine(gpu_engine_factory, box, v, rc=7.0, skin=1.0, sz=(32, 32, 32), order=5, e3b=True,
                                   dt=1.0)
        e.teams_set(team)
        return e, flags

    e, flags = make(start_velocities(orc, box, seed=9))
    e.option("graph", graph)

    def oracle_list():
        x, _ = e.get_system()
        return (x, *oracle_rows_by_id(orc, x, box["lo"], L, 8.0, excl=excl, brute=False)[:2])

    for _ in range(2):
        e.run(70, flags)
        e.nlist_update(force=True)
        x, oc, orows = oracle_list()
        read = e.pair_entries_read()
        assert e.nlist_totals()[0] == int(oc.sum())  # completed, then partial again by the run
        assert e.pair_entries_read() == read and read[0] < 0.75 * oc.sum()
    v = e.get_system()[1]
    g, _ = make(v)  # a reader of the list: whole rows from then on
    g.option("graph", graph)
    g.set_positions(x)
    for _ in range(2):
        g.nlist_update(force=True)
        assert_same_lists(*g.nlist_get(), oc, orows)
    for k in (e, g):
        k.compute(flags)
    assert np.array_equal(e.forces(), g.forces())
    g.close()
    # LJ between every pair of types: every part of every row is read now
    rc2 = np.full((3, 3), 49.0)
    eps24, sig6 = np.full((3, 3), 24 * 0.05), np.full((3, 3), 1.0)
    f, _ = make(np.zeros_like(box["x"]))
    f.set_positions(x)
    out = []
    for k in (e, f):
        k.lj_set(rc2, eps24, sig6)
        k.compute(PAIR | PPPM | E3B)
        out.append(k.forces())
        k.close()
    assert np.array_equal(out[0], out[1])


def test_box_turned_on_its_side(orc, gpu_engine_factory):
    """An elongated box turned on one engine: 6 x 6 x 24 cells (36 columns),
    then 12 x 6 x 12 (as many cells, 72 columns) and back."""
    say("elongated box turned on its side")
    rng = np.random.default_rng(7)
    n, rlist = 1500, 10.0
    q = np.where(rng.random(n) < 0.4, 0.3, 0.0)
    u = rng.uniform(0, 1, (n, 3))
    e = None
    for L, cells in ((np.array([31.0, 31.0, 62.0]), (6, 6, 24)), (np.array([62.0, 31.0, 31.0]), (12, 6, 12)),
                     (np.array([31.0, 31.0, 62.0]), (6, 6, 24))):
        x = u * L
        if e is None:
            e = _list_engine(gpu_engine_factory, x, L, rlist, 1.0, q=q)
        else:
            e.set_box(np.zeros(3), L)
            e.set_positions(x)
        e.nlist_update(force=True)
        assert tuple(e.nlist_stats()["cells"]) == cells
        gc, grows = e.nlist_get()
        oc, orows, _ = oracle_rows_by_id(orc, x, np.zeros(3), L, rlist, brute=True)
        assert_same_lists(gc, grows, oc, orows)
    e.close()


@pytest.mark.parametrize("first,then", [(64, 16), (16, 64)])
def test_list_read_after_a_capture_of_another_build(orc, gpu_engine_factory, first, then):
    """Wave builds keep the exclusion partners by id, team builds by index.
    Steps captured for the other kind, none of which built a list, leave the
    current list's rows as their own build left them: the list read back has
    the tags of the exclusions."""
    say(f"list of a {first}-lane build read back after captured steps of {then} lanes")
    from md_engine_amd import systems
    from test_gpu_water_md import start_velocities, water_md_engine

    box = systems.tip4p2005_box(343, seed=36, min_sep=1.8)
    e, flags = water_md_engine(gpu_engine_factory, box, start_velocities(orc, box, seed=9), rc=7.0, skin=1.0,
                               sz=(32, 32, 32), order=5, e3b=False, dt=0.5)
    e.teams_set(build=first)
    # the records in an order of cells, not of ids
    e.compute(flags)
    before = e.nlist_stats()["rebuilds"]
    e.option("graph", 1)
    e.teams_set(build=then)
    e.run(2, flags)
    # the run's start builds anew (rigid molecules placed); the steps do not
    built = e.nlist_stats()["rebuilds"] - before
    e.teams_set(build=first)
    e.nlist_update(force=True)
    e.teams_set(build=then)
    x, _ = e.get_system()
    before = e.nlist_stats()["rebuilds"]
    e.run(2, flags)
    assert e.nlist_stats()["rebuilds"] == before and built <= 1
    gc, grows = e.nlist_get()
    excl = orc.exclusions_bfs(len(x), systems.water_bonds(box["mol"]))
    oc, orows, _ = oracle_rows_by_id(orc, x, box["lo"], box["L"], 8.0, excl=excl, brute=False)
    assert_same_lists(gc, grows, oc, orows)
    e.close()
