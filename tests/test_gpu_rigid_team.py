"""The rigid first half with four lanes a molecule (up to 16,384 molecules) and
with one (beyond): molecules without interactions move alike, bit for bit, in a system
on either side of the line, and where the last workgroup is not full."""
import sys

import numpy as np
import pytest

from md_engine_amd import systems

from test_gpu_water_md import G, min_image_diff, start_velocities

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def free_molecules(make, box, v, nmol, steps):
    from md_engine_amd import PAIR

    mol = box["mol"][:nmol]
    n = 4 * nmol  # the generator numbers a molecule's sites together
    mass = box["mass"][:n]
    e = make()
    e.set_system(box["x"][:n], box["lo"], box["L"], v=v[:n], types=box["type"][:n],
                 inv_mass=np.where(mass > 0, 1.0 / np.maximum(mass, 1e-30), 0.0))
    e.exclusions_from_bonds(systems.water_bonds(mol))
    e.nlist_config(4.0, 1.0)
    e.lj_set(np.full((3, 3), 9.0), np.zeros((3, 3)), np.ones((3, 3)))
    e.rigid_set(mol, G["mO"], G["mH"], G["dOH"], G["dHH"], G["gamma"])
    e.integrator_set(1.0, systems.REAL_FTM_TO_V)
    e.run(steps, PAIR)
    out = e.get_system()
    e.close()
    return out


def test_teams_of_four_match_one_lane(orc, gpu_engine_factory):
    say("rigid first half: 1, 33, 16384 molecules (four lanes) and 16385 (one)")
    box = systems.tip4p2005_box(16385, seed=1)
    v = start_velocities(orc, box, seed=4)
    steps = 30
    x1, v1 = free_molecules(gpu_engine_factory, box, v, 16385, steps)
    d = min_image_diff(x1[1::4], x1[0::4], box["L"])
    assert np.allclose(np.linalg.norm(d, axis=1), G["dOH"], atol=1e-8)
    assert np.abs(min_image_diff(x1[0::4], box["x"][0::4], box["L"])).max() > 0.05
    for nmol in (1, 33, 16384):
        x4, v4 = free_molecules(gpu_engine_factory, box, v, nmol, steps)
        assert np.array_equal(x4, x1[: 4 * nmol])
        assert np.array_equal(v4, v1[: 4 * nmol])


@pytest.mark.parametrize("sizes,baro", [((33, 16384, 16385), False), ((33, 12288, 12289), True)])
def test_batch_across_the_lines(orc, gpu_engine_factory, sizes, baro):
    """A batch with replicas on both sides of a size rule (four lanes or one a
    molecule; the barostat step within the second half or as launches of its
    own) takes one side for all of them: one launch a kernel, and each replica
    as it runs alone."""
    from md_engine_amd import PAIR, run_batch

    say(f"batch of {sizes} molecules, barostat {baro}")
    box = systems.tip4p2005_box(max(sizes), seed=1)
    v = start_velocities(orc, box, seed=4)

    def make(nmol):
        n, mass = 4 * nmol, box["mass"][: 4 * nmol]
        e = gpu_engine_factory()
        e.set_system(box["x"][:n], box["lo"], box["L"], v=v[:n], types=box["type"][:n],
                     inv_mass=np.where(mass > 0, 1.0 / np.maximum(mass, 1e-30), 0.0))
        e.exclusions_from_bonds(systems.water_bonds(box["mol"][:nmol]))
        e.nlist_config(4.0, 1.0)
        eps24, sig6 = systems.water_lj_tables()
        e.lj_set(np.full((3, 3), 9.0), eps24, sig6)
        e.rigid_set(box["mol"][:nmol], G["mO"], G["mH"], G["dOH"], G["dHH"], G["gamma"])
        e.integrator_set(1.0, systems.REAL_FTM_TO_V)
        if baro:
            e.barostat(True, 1.0, 1000.0, 1, mvv_to_eng=systems.REAL_MVV_TO_ENG)
        e.option("graph", 1)
        return e

    batch = [make(m) for m in sizes]
    run_batch(batch, 24, PAIR)
    assert batch[0].batch_merged()
    for e, m in zip(batch, sizes):
        alone = make(m)
        alone.run(24, PAIR)
        for a, b in zip((*e.get_system(), e.get_box()[1]), (*alone.get_system(), alone.get_box()[1])):
            assert np.array_equal(a, b), m
        alone.close()
    for e in batch:
        e.close()
