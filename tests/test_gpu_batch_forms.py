"""Batches in the long plain step (time_step_factor above 0.25) and mixed ones, in which
members that take the short step alone are taken along in the long one: every member
ends bit-equal to its own run, whatever the schedule, and whatever it did before it
joined the batch."""
import numpy as np
import pytest

from amca3d_amd import decks
from test_gpu_batch import _same

pytestmark = pytest.mark.gpu

# (edge or shape, seed, Tdot, density): ten members, so that the maps are rebuilt as
# some of them finish
MEMBERS = [((12, 12, 12), 3, -25.0, 8e15), ((40, 40, 40), 0, -1800.0, 1e15),
           ((20, 9, 33), 7, -300.0, 4e15), ((33, 33, 33), 11, -60.0, 2e15),
           ((16, 16, 16), 5, -1000.0, 6e15), ((27, 27, 27), 2, -150.0, 1.5e15),
           ((18, 18, 18), 13, -40.0, 5e15), ((24, 24, 24), 17, -700.0, 3e15),
           ((5, 70, 6), 19, -90.0, 7e15), ((30, 30, 30), 23, -2500.0, 1e15)]
LONG, MIXED = [0.3] * 10, [0.2, 0.3, 0.2, 0.2, 1.0, 0.25, 0.26, 0.2, 0.3, 0.2]


def _text(member, tsf):
    (nx, ny, nz), seed, tdot, rho = member
    return decks.plain_deck(nx, ny, nz, 2e-6, bulk=(rho, 3.0, 1.0), Tdot=tdot, T0=-0.2,
                            termination_time=1.0, time_step=1e-3, random_seed=seed,
                            time_step_factor_ca=tsf)


def _state(s):
    d = s.domain
    o = d.download()
    return dict(c=d.counters(), ori=o["ori"], gid=o["gid"], env=o["env"], log=d.read_log())


@pytest.fixture(scope="module")
def singles():
    import amca3d_amd as amca
    memo = {}

    def get(member, tsf):
        if (member, tsf) not in memo:
            with amca.Simulation(_text(member, tsf)) as s:
                s.initialize()
                s.domain.enable_log(100000)
                s.run()
                memo[member, tsf] = _state(s)
        return memo[member, tsf]
    return get


def _check(amca, singles, factors, schedule=None, autotune=False, before=None, calls=-1):
    from amca3d_amd.batch import Batch
    sims = [amca.Simulation(_text(m, f)).initialize() for m, f in zip(MEMBERS, factors)]
    for i, s in enumerate(sims):
        s.domain.enable_log(100000)
        if before:
            s.run(before[i % len(before)])
    b = Batch([s.domain for s in sims])
    if schedule:
        b.set_schedule(**schedule)
    if autotune:
        b.autotune(trial_graphs=1, rounds=2)
    for _ in range(20000):
        if b.run(calls)["finished"] == len(sims):
            break
    b.close()
    for s, m, f in zip(sims, MEMBERS, factors):
        a = singles(m, f)
        assert a["c"]["done"] == 1
        _same(a, _state(s))
        s.close()


@pytest.mark.parametrize("factors", [LONG, MIXED], ids=["long", "mixed"])
@pytest.mark.parametrize("schedule", [
    None,
    # one step per replay: the maps are rebuilt at once each time four more have finished
    dict(list_blocks=64, emit_blocks=64, min_blocks=1, interleave=1, steps_per_graph=1),
    dict(list_blocks=6, emit_blocks=7, min_blocks=1, interleave=1, steps_per_graph=3),
    # above four blocks per CU: a quarter of one budget, four per CU of the other
    dict(list_blocks=4096, emit_blocks=16384, min_blocks=8, interleave=0, steps_per_graph=64),
])
def test_batch_equals_single_runs(amca, singles, factors, schedule):
    _check(amca, singles, factors, schedule)


@pytest.mark.parametrize("factors", [LONG, MIXED], ids=["long", "mixed"])
def test_after_autotune(amca, singles, factors):
    _check(amca, singles, factors, autotune=True)


def test_autotune_of_the_short_step_leaves_the_claim_budget(amca):
    """The short step's claims run on the grid of emit_blocks: the claim budget stays the
    one tried for all kernels together."""
    from amca3d_amd.batch import Batch
    sims = [amca.Simulation(_text(m, 0.2)).initialize() for m in MEMBERS]
    for s in sims:
        s.domain.counters()
    b = Batch([s.domain for s in sims])
    cus = b.schedule()["list_blocks"] // 16
    for _ in range(3):
        c = b.autotune(trial_graphs=1, rounds=1)
        assert c["list_blocks"] in [2 * cus, 16 * cus, 64 * cus]
        assert c["emit_blocks"] in [cus * e for e in (1, 2, 4, 8, 16, 64, 128)]
        assert b.schedule() == c
    b.close()
    for s in sims:
        s.close()


def test_members_with_steps_of_their_own(amca, singles):
    """Members that ran in their own form first, to different steps, join a long batch."""
    _check(amca, singles, MIXED, dict(steps_per_graph=5), before=[1, 0, 37, 150, 16])


def test_without_graphs_one_replay_per_call(amca, singles, monkeypatch):
    monkeypatch.setenv("AMCA_BATCH_GRAPHS", "0")
    _check(amca, singles, MIXED, dict(steps_per_graph=4), calls=1)


def test_member_matches_oracle(amca, oracle, singles):
    for m, tsf in ((MEMBERS[2], 0.2), (MEMBERS[3], 0.3), (MEMBERS[8], 0.3)):
        (nx, ny, nz), seed, tdot, rho = m
        r = oracle.run_plain(oracle.plain_params(
            nx=nx, ny=ny, nz=nz, h=2e-6, nv=rho, dTv_mean=3.0, dTv_sd=1.0, seed=seed, Tdot=tdot,
            max_dt=1e-3, final_time=1.0, tsf=tsf), want_grains=False)
        a = singles(m, tsf)
        assert a["c"]["step"] == r["n_steps"]
        np.testing.assert_array_equal(a["ori"], r["ori"])
        np.testing.assert_array_equal(a["gid"], r["gid"])
