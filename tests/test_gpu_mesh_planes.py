"""The mesh solve's in-place passes at the edges of their dispatch: every line
length on every axis, planes on both sides of the line between
512 and 1,024 threads, few and many column groups; against the FP64 oracle's
P3M and the library transforms."""
import sys

import numpy as np
import pytest

from md_engine_amd import systems

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("sz", [(32, 128, 32), (128, 32, 32), (64, 32, 128), (64, 64, 64), (64, 64, 128),
                                (64, 128, 64), (128, 128, 64), (128, 128, 128)])
def test_in_place_planes(orc, gpu_engine_factory, sz):
    say(f"in-place mesh planes {sz}")
    from md_engine_amd._lib import ENERGY, PPPM, VIRIAL
    from test_gpu_parity import FORCE_RMSE, rel_rmse

    box = systems.tip4p2005_box(216, seed=15)
    n, order, rc, qqr, alpha = len(box["x"]), 3, 7.0, systems.REAL_QQR_TO_ENG, 0.3
    e = gpu_engine_factory()
    e.set_system(box["x"], box["lo"], box["L"], q=box["q"], types=box["type"], inv_mass=np.ones(n))
    e.nlist_config(rc + 1.0, 1.0)
    e.pppm_set(sz, order, rc, qqr, alpha=alpha)
    G = orc.pppm_green(box["L"], np.array(sz), alpha, order)
    ref = orc.pppm(box["x"], box["q"], box["lo"], box["L"], np.array(sz), order, qqr, alpha,
                   orc.total_q2(box["q"], qqr), G, energy=True, virial=True)
    out = {}
    for mode in (1, 0):
        e.option("p3m_fft", mode)
        e.compute(PPPM)
        f0 = e.forces()
        e.compute(PPPM | ENERGY | VIRIAL)  # from the cleared charge mesh, with the sums' waves
        assert e.pppm_paths()[2] == mode
        f = e.forces()
        en, vk = e.energies()
        assert np.array_equal(f0, f)
        out[mode] = f, en[1], vk
        assert rel_rmse(f, ref["f"]) <= FORCE_RMSE
        assert en[1] == pytest.approx(ref["energy"], rel=1e-5)
        assert np.allclose(vk, ref["virial"], rtol=1e-4, atol=1e-4 * np.abs(ref["virial"]).max())
    # two FP32 transforms of at most 21 halvings each: 42 roundings of 6e-8
    d = [rel_rmse(out[m][0], ref["f"]) for m in (0, 1)]
    say(f"force RMSE library {d[0]:.2e}, in place {d[1]:.2e}")
    assert max(d) <= 2.5e-6
    e.close()


def test_batch_of_several_meshes(gpu_engine_factory):
    """Replicas whose meshes lie on both sides of the passes' size rules run
    the same kernels in a batch: one launch a kernel, and each as alone."""
    from md_engine_amd import PPPM, run_batch
    from test_gpu_water_md import water_md_engine

    say("batch of 32^3, 64^3, 64 x 64 x 128 and 128^3 meshes")
    box = systems.tip4p2005_box(512, seed=15)
    meshes = [(32, 32, 32), (64, 64, 64), (64, 64, 128), (128, 128, 128)]

    def make(sz):
        e, _ = water_md_engine(gpu_engine_factory, box, np.zeros_like(box["x"]), rc=7.0, skin=1.0, sz=sz, order=3,
                               e3b=False, dt=1.0)
        for k, v in (("graph", 1), ("p3m_spread", 0), ("p3m_gather", 1)):  # whatever the tiles of a mesh hold
            e.option(k, v)
        return e

    batch = [make(sz) for sz in meshes]
    run_batch(batch, 20, PPPM)
    assert batch[0].batch_merged()
    for e, sz in zip(batch, meshes):
        alone = make(sz)
        alone.run(20, PPPM)
        assert e.pppm_paths()[2] == alone.pppm_paths()[2] == 1
        for a, b in zip(e.get_system(), alone.get_system()):
            assert np.array_equal(a, b), sz
        alone.close()
    for e in batch:
        e.close()
