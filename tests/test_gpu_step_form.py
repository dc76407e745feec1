"""The choice between the short and the long plain step as a run goes: dense grains,
whose fresh envelopes often capture in the step that made them, take the long step,
and the results are the same on both sides of every change."""
import numpy as np
import pytest

from amca3d_amd import decks
from test_gpu_plain import case, compare

pytestmark = pytest.mark.gpu

# 96^3 cells: dense grains of a large truncation, of which some thousands a step are
# wave-1 grains beside a wave-1 claim; and sparse ones, of which next to none are
DENSE = dict(nx=96, ny=96, nz=96, h=2e-6, bulk=(1e16, 3.0, 1.0), Tdot=-200.0, time_step=1e-4,
             max_half_diagonal_length=12.0, seed=5)
SPARSE = dict(nx=96, ny=96, nz=96, h=2e-6, bulk=(5e13, 3.0, 1.0), Tdot=-200.0, time_step=1e-4,
              seed=5)


def _run(amca, text, timing, chunks=(-1,)):
    s = amca.Simulation(text).initialize()
    d = s.domain
    d.enable_log(1 << 16)
    if timing:
        d.enable_timing(True)
    for n in chunks:
        c = s.run(n)
    out = d.download()
    out["grains"] = d.download_grains()
    out["log"] = d.read_log()
    out["counters"] = c
    out["initial_sites"] = s.initial_sites()
    kt = d.kernel_times() if timing else None
    s.close()
    return out, kt


@pytest.fixture(scope="module")
def dense_oracle(oracle):
    return oracle.run_plain(oracle.plain_params(**case(**DENSE)[1]))


@pytest.mark.parametrize("timing", [False, True])
def test_dense_growth_takes_the_long_step(amca, oracle, dense_oracle, timing):
    text, prm = case(**DENSE)
    g, kt = _run(amca, text, timing)
    compare(oracle, prm, g, dense_oracle)
    if timing:
        # k_compact is launched by the long step only
        n = g["counters"]["step"]
        assert 0 < kt["k_compact"][1] < n and kt["k_tail"][1] >= n


def test_sparse_growth_stays_with_the_short_step(amca):
    _, kt = _run(amca, case(**SPARSE)[0], True)
    assert kt["k_compact"][1] == 0 and kt["k_tail"][1] > 0


def test_many_sites_start_with_the_long_step(amca):
    """Sites enough for a nucleation burst: the long step before any of them nucleates."""
    kw = dict(DENSE, nx=192, ny=192, nz=192, bulk=(2e15, 3.0, 1.0), max_half_diagonal_length=None)
    _, kt = _run(amca, case(**kw)[0], True, [5])
    assert kt["k_compact"][1] == kt["k_tail"][1] == 5


def test_form_changes_between_calls(amca, oracle, dense_oracle):
    """The same run in pieces of uneven length, single steps among them."""
    text, prm = case(**DENSE)
    g, _ = _run(amca, text, False, [3, 17] + [1] * 20 + [40, 5, 33, -1])
    compare(oracle, prm, g, dense_oracle)


def test_fixed_steps_change_form(amca, oracle, dense_oracle):
    import ctypes as C

    from amca3d_amd._lib import load
    text, prm = case(**DENSE)
    s = amca.Simulation(text).initialize()
    d = s.domain
    d.enable_log(1 << 16)
    assert load().amca_domain_run_fixed(d.h, C.c_int64(dense_oracle["n_steps"] + 70)) == 0
    out = d.download()
    out["grains"] = d.download_grains()
    out["log"] = d.read_log()
    out["counters"] = d.counters()
    out["initial_sites"] = s.initial_sites()
    compare(oracle, prm, out, dense_oracle)
    s.close()


def test_dense_batch_changes_form(amca, oracle, dense_oracle):
    """A batch that goes from the short to the long step and, as its dense member
    finishes, may come back: every member ends as its own run does."""
    from amca3d_amd.batch import Batch
    texts = [case(**DENSE)[0]] + [
        decks.plain_deck(e, e, e, 2e-6, bulk=(rho, 3.0, 1.0), Tdot=t, time_step=1e-4,
                         termination_time=17.81, random_seed=e)
        for e, rho, t in ((40, 1e15, -300.0), (33, 2e15, -60.0), (64, 5e13, -200.0),
                          (20, 4e15, -100.0), (27, 1e14, -150.0))]
    singles = [_run(amca, t, False)[0] for t in texts]
    for steps in (1, 16):
        sims = [amca.Simulation(t).initialize() for t in texts]
        for s in sims:
            s.domain.enable_log(1 << 16)
        b = Batch([s.domain for s in sims])
        b.set_schedule(steps_per_graph=steps)
        assert b.run()["finished"] == len(sims)
        b.close()
        for s, w in zip(sims, singles):
            d = s.domain
            o = d.download()
            for k in ("ori", "gid", "env"):
                assert np.array_equal(o[k], w[k]), k
            for k in ("step", "n_grains", "n_orient", "n_active", "time"):
                assert d.counters()[k] == w["counters"][k], k
            log = d.read_log()
            for k in ("dt", "n_captured", "n_active_after", "n_wave1", "max_wave"):
                assert np.array_equal(log[k], w["log"][k]), k
            s.close()
    assert np.array_equal(singles[0]["gid"], dense_oracle["gid"])
