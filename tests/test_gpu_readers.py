"""State and forces read from several threads at once: the arrays are packed by
atom id in a buffer of the context, which one reader holds at a time."""
import threading

import numpy as np
import pytest

from md_engine_amd import PAIR, systems

pytestmark = pytest.mark.gpu


def test_concurrent_readers(gpu_engine_factory):
    print("four threads reading state and forces", flush=True)
    x, L, lo = systems.fcc_lj(20, 0.8442)
    n = len(x)
    e = gpu_engine_factory()
    e.set_system(x, lo, L, v=systems.maxwell_boltzmann(np.ones(n), 1.2, seed=4), inv_mass=np.ones(n))
    e.lj_set([[6.25]], [[24.0]], [[1.0]])
    e.nlist_config(2.8, 0.3)
    e.integrator_set(0.005, 1.0)
    e.run(20, PAIR)
    (x0, v0), f0 = e.get_system(), e.forces()
    bad = []

    def reader(k):
        for _ in range(40):
            if k % 2:
                x1, v1 = e.get_system()
                ok = np.array_equal(x1, x0) and np.array_equal(v1, v0)
            else:
                ok = np.array_equal(e.forces(), f0)
            if not ok:
                bad.append(k)

    threads = [threading.Thread(target=reader, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    e.close()
    assert not bad


def test_concurrent_list_readers(gpu_engine_factory):
    """The list read back from several threads: the first completes the rows
    that steps leave out, the others wait for it."""
    print("four threads reading the list", flush=True)
    box = systems.tip4p2005_box(343, seed=36, min_sep=1.8)
    from test_gpu_water_md import water_md_engine

    e, flags = water_md_engine(gpu_engine_factory, box, np.zeros_like(box["x"]), rc=7.0, skin=1.0, sz=(32, 32, 32),
                               order=5, e3b=True, dt=1.0)
    e.compute(flags)
    got = [None] * 4

    def reader(k):
        got[k] = e.nlist_totals() if k == 0 else e.nlist_get()

    threads = [threading.Thread(target=reader, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    e.nlist_update(force=True)
    counts, rows = e.nlist_get()
    e.close()
    assert got[0][0] == counts.sum()
    for c, r in got[1:]:
        assert np.array_equal(c, counts)
        assert all(np.array_equal(a, b) for a, b in zip(r, rows))
