"""The Nose-Hoover half step at its shortest and longest chain (2 links; 64, whose
state is longer than the wave that stages it) against the FP64 restatement."""
import sys

import numpy as np
import pytest

from md_engine_amd import systems

from test_gpu_water_md import min_image_diff, start_velocities, water_md_engine

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("chain", [2, 64])
def test_chain_lengths_match_oracle(orc, gpu_engine_factory, chain):
    say(f"Nose-Hoover chain of {chain} links vs oracle")
    from oracle.thermostat import water_md_nh

    box = systems.tip4p2005_box(216, seed=25, min_sep=1.8)
    v = start_velocities(orc, box, seed=8) * np.sqrt(350.0 / 298.0)
    kw = dict(rc=7.0, skin=1.0, sz=(32, 32, 32), order=5)
    e, flags = water_md_engine(gpu_engine_factory, box, v, e3b=False, dt=1.0, **kw)
    kb, mvv = systems.REAL_BOLTZ, systems.REAL_MVV_TO_ENG
    e.nose_hoover(True, 298.0, 20.0, chain, kb, mvv)
    e.run(20, flags)
    xg, vg = e.get_system()
    st = e.nose_hoover_state(chain)
    xo, vo, ch = water_md_nh(box, v, 20, 298.0, 20.0, chain=chain, dt=1.0, e3b_on=False, **kw)
    so = ch.state()
    e.close()
    dx = np.abs(min_image_diff(xg, xo, box["L"])).max()
    heavy = box["mass"] > 0
    rel_v = np.abs(vg[heavy] - vo[heavy]).max() / np.abs(vo[heavy]).max()
    say(f"dx {dx:.2e} A, rel v {rel_v:.2e}")
    # the bounds of the 10-link test of 50 steps
    assert dx < 1e-5, dx
    assert rel_v < 1e-4, rel_v
    # chain velocities, forces, masses and positions, sum m v^2, last scale
    for k, name in enumerate(("v", "G", "Q", "xi")):
        a, b = st[k * chain : (k + 1) * chain], so[k * chain : (k + 1) * chain]
        err = np.abs(a - b).max() / np.abs(b).max()
        assert err < 1e-4, (name, err)
    assert st[4 * chain] == pytest.approx(so[4 * chain], rel=1e-5)
    assert st[4 * chain + 1] == pytest.approx(so[4 * chain + 1], rel=1e-9)
