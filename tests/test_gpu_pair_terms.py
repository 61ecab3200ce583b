"""Pair forces where neighbouring atoms need different terms: a wave takes the
code of LJ, of Coulomb or of both for a row part by what any of its atoms needs
there, so atoms with charge and LJ, with one of them and with neither share
waves here.  Against the FP64 oracle; forces and energies to the bars of the
other pair tests (FP32 separations in a 20 A box, 1e-4 of the RMS force)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("flags", ["force", "energy"])
@pytest.mark.parametrize("kinds", ["one_type", "lj_of_some", "no_lj_charged", "no_charges"])
def test_atoms_of_mixed_terms(orc, gpu_engine_factory, kinds, flags):
    from md_engine_amd._lib import ENERGY, PAIR, VIRIAL
    from test_gpu_parity import assert_same_lists, oracle_rows_by_id, rel_rmse

    say(f"pair terms: {kinds}, {flags}")
    rng = np.random.default_rng(17)
    m = 10
    g = np.stack(np.meshgrid(*3 * [np.arange(m)], indexing="ij"), -1).reshape(-1, 3)[:-7]
    L, lo = np.full(3, 20.0), np.zeros(3)
    x = (g + 0.5) * 2.0 + rng.uniform(-0.3, 0.3, g.shape)
    n = len(x)  # 993: the last wave is not full
    T = 1 if kinds == "one_type" else 3
    types = rng.integers(0, T, n).astype(np.int32)
    q = rng.uniform(-1, 1, n) * (rng.random(n) < 0.6)
    sig, eps = np.array([1.6, 1.9, 1.7])[:T], np.array([0.3, 0.0, 0.2])[:T]
    if kinds == "no_lj_charged":  # the water pattern: LJ only between charge-free atoms
        q[types == 0] = 0.0
        eps = np.array([0.3, 0.0, 0.0])
    if kinds == "no_charges":
        q[:] = 0.0
    eps24 = 24.0 * np.sqrt(np.outer(eps, eps))
    sig6 = (0.5 * (sig[:, None] + sig[None, :])) ** 6
    rc, skin, alpha, qqr = 6.0, 0.7, 0.35, 332.06
    rc2 = np.full((T, T), rc * rc)
    bonds = np.stack([np.arange(0, n - 1, 3), np.arange(1, n, 3)], 1)
    e = gpu_engine_factory()
    e.set_system(x, lo, L, q=q, types=types, inv_mass=np.ones(n))
    e.exclusions_from_bonds(bonds)
    e.nlist_config(rc + skin, skin)
    e.lj_set(rc2, eps24, sig6)
    e.pppm_set((32, 32, 32), 5, rc, qqr, alpha=alpha)
    e.ewald_real_set(True, -1.0, qqr, rc)
    e.compute(PAIR | (ENERGY | VIRIAL if flags == "energy" else 0))
    f = e.forces()
    oc, orows, xw = oracle_rows_by_id(orc, x, lo, L, rc + skin, excl=orc.exclusions_bfs(n, bonds), brute=False)
    fo, eo, vo = orc.pair(xw, q, types, L, oc, orows, rc2, eps24, sig6, with_charge=True, alpha=alpha, qqr=qqr, rq=rc)
    assert rel_rmse(f, fo) <= 1e-4
    if flags == "energy":
        en, vir = e.energies()
        assert en[0] == pytest.approx(eo.sum(), rel=1e-5, abs=1e-5 * np.abs(eo).sum())
        assert np.allclose(vir, vo, rtol=1e-5, atol=1e-5 * np.abs(vo).max())
    assert_same_lists(*e.nlist_get(), oc, orows)
    e.close()
