"""The long plain step (time_step_factor above 0.25, or dense sites) against the CPU
oracle on grids of many compaction, list and id-scan blocks (many bricks per block:
test_gpu_batch_forms.py, whose small budgets give a domain one block): fields, envelopes, sites and the step log to the bit, and the
kernels that only the long step launches counted."""
import numpy as np
import pytest

from amca3d_amd import decks
from test_gpu_plain import compare
from test_gpu_step_form import _run

pytestmark = pytest.mark.gpu


def _case(shape, tsf, density, max_steps=-1):
    nx, ny, nz = shape
    text = decks.plain_deck(nx, ny, nz, 2e-6, surface=(1e9, 1.0, 0.5), surface_faces="z_min",
                            bulk=(density, 3.0, 1.0), Tdot=-200.0, time_step=1e-4,
                            termination_time=1.0, random_seed=7, time_step_factor_ca=tsf)
    prm = dict(nx=nx, ny=ny, nz=nz, h=2e-6, ns=1e9, dTs_mean=1.0, dTs_sd=0.5, surface_mode=1,
               nv=density, dTv_mean=3.0, dTv_sd=1.0, seed=7, Tdot=-200.0, max_dt=1e-4,
               final_time=1.0, tsf=tsf, max_steps=max_steps)
    return text, prm


# 96^3 is 27 id-scan blocks at most and 245 compaction blocks, 144^3 92 and 792
@pytest.mark.parametrize("shape,tsf,density,steps", [
    ((96, 96, 96), 0.3, 5e13, -1),
    ((131, 97, 67), 0.3, 2e14, -1),
    ((67, 131, 97), 0.8, 5e13, -1),
    ((144, 144, 144), 0.3, 5e13, 220),
    # the default factor, in the long step from the start by its 4.8e4 sites
    ((144, 144, 144), 0.2, 2e15, -1),
])
def test_long_step_parity(amca, oracle, shape, tsf, density, steps):
    text, prm = _case(shape, tsf, density, steps)
    g, kt = _run(amca, text, True, (steps,))
    r = compare(oracle, prm, g)
    if tsf > 0.25:
        assert kt["k_compact"][1] == kt["k_tail"][1] > 0
    else:
        # long at least while more than 3000 sites are live (the choice is made from
        # counters of the same step or earlier ones, which hold as many or more); captures
        # by grains captured in the same step in many of these
        many = int((g["log"]["n_sites"] > 3000).sum())
        assert kt["k_compact"][1] >= many > 100
        assert (g["log"]["max_wave"] >= 2).sum() > 10
    # without events, from graphs
    g2, _ = _run(amca, text, False, (steps,))
    for k in ("ori", "gid", "env"):
        assert np.array_equal(g[k], g2[k]), k
