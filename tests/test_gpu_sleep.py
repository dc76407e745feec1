"""Sleeping grains and the two forms of the plain step against the CPU oracle:
grids with partial bricks on every axis, growth per step on both sides of the
line between the short and the long step (time_step_factor 0.25), runs across
several refresh steps, and downloads in the middle of sleeps (the envelopes of
sleeping grains are worked out for them)."""
import numpy as np
import pytest

from amca3d_amd import decks
from test_gpu_plain import compare, run_gpu

pytestmark = pytest.mark.gpu


def _case(shape, tsf, max_dt, tdot=-200.0, density=2e14, seed=3):
    nx, ny, nz = shape
    text = decks.plain_deck(nx, ny, nz, 2e-6, bulk=(density, 3.0, 1.0), Tdot=tdot,
                            time_step=max_dt, termination_time=10.0, random_seed=seed,
                            time_step_factor_ca=tsf)
    prm = dict(nx=nx, ny=ny, nz=nz, h=2e-6, nv=density, dTv_mean=3.0, dTv_sd=1.0, seed=seed,
               Tdot=tdot, max_dt=max_dt, final_time=10.0, tsf=tsf)
    return text, prm


# 0.25: the short step's largest growth; above it the long step, whose fresh grains
# capture in the same step often
@pytest.mark.parametrize("tsf", [0.05, 0.25, 0.26, 0.9, 2.5])
@pytest.mark.parametrize("shape", [(1, 1, 9), (3, 4, 5), (17, 30, 6), (64, 1, 33), (41, 38, 35)])
def test_both_step_forms(amca, oracle, shape, tsf):
    # dt is the growth's (max_dt never binds once grains grow fast)
    text, prm = _case(shape, tsf, 2e-3, density=5e14)
    compare(oracle, prm, run_gpu(amca, text))


@pytest.mark.parametrize("tsf", [0.2, 0.3])
def test_refresh_steps(amca, oracle, tsf):
    """A run of several thousand steps: every active grain wakes at steps 2048, 4096, ..."""
    text, prm = _case((23, 18, 21), tsf, 5e-6)
    r = compare(oracle, prm, run_gpu(amca, text))
    assert r["n_steps"] > 2 * 2048 + 100


@pytest.mark.parametrize("tsf", [0.2, 0.3])
def test_downloads_between_steps(amca, oracle, tsf):
    text, prm = _case((23, 18, 21), tsf, 5e-6)
    s = amca.Simulation(text).initialize()
    at = 0
    for stop in (1500, 2047, 2048, 2049, 2500, 4097):
        c = s.run(stop - at)
        at = stop
        g = s.domain.download()
        r = oracle.run_plain(oracle.plain_params(**dict(prm, max_steps=stop)))
        assert c["step"] == r["n_steps"] and c["n_active"] == r["n_active"]
        assert np.array_equal(g["gid"], r["gid"]) and np.array_equal(g["ori"], r["ori"])
        env = np.zeros((len(r["ori"]), 4))
        env[r["grain_cell"]] = r["env"]
        assert np.array_equal(g["env"][r["grain_cell"]], env[r["grain_cell"]])
    s.close()


def test_growth_past_the_clock_span(amca, oracle):
    """A few seeds in a long bar: the front crosses more than the growth clock's 60
    cells, so the clock restarts between the regular refresh steps."""
    text, prm = _case((220, 5, 4), 0.2, 2e-3, density=6e13)
    r = compare(oracle, prm, run_gpu(amca, text))
    st = r["steps"][:r["n_steps"]]
    # the growth of each step in cells: dt times the velocity at the step's undercooling
    # (T0 = -0.2 K, the deck's a1 and a2); the clock restarts past 60
    p = oracle.plain_params(**prm)
    u = p.Tm - (p.T0 + p.Tdot * st["time_before"])
    clock, restarts = 0.0, []
    for i, g in enumerate(st["dt"] * np.maximum(p.a1 * u + p.a2 * u * u, 0.0) / p.h):
        clock += g
        if clock > 60.0:
            clock = 0.0
            restarts.append(i)
    # before the first regular refresh step after step 0, with captures beyond the last
    assert r["n_steps"] < 2048 and len(restarts) >= 5
    assert st["n_captured"][restarts[-1] + 1:].sum() > 100


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 62, 6), (62, 3, 2), (63, 5, 7), (130, 9, 4)])
def test_device_fields_match_the_downloads(amca, shape):
    """The by-cell and by-id layouts on the device, part-way through a run, on grids
    around the 16-brick rows that their kernel takes: the same values as the
    downloads of fields, envelopes and grains."""
    import ctypes as C

    from amca3d_amd._lib import load
    memcpy = load().hipMemcpy  # of the runtime that the library is linked to
    memcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]

    def host(ptr, shape, dtype):
        a = np.empty(shape, dtype)
        assert memcpy(a.ctypes.data, ptr.value, a.nbytes, 2) == 0  # device to host
        return a

    text, _ = _case(shape, 0.2, 2e-3, density=2e15)
    s = amca.Simulation(text).initialize()
    n = s.run(30)["n_grains"]
    d = s.domain
    f = d.download()
    o, g, e = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert load().amca_domain_device_fields(d.h, C.byref(o), C.byref(g), C.byref(e), None) == 0
    ng = f["gid"].size
    for p, want in ((o, f["ori"]), (g, f["gid"])):
        assert np.array_equal(host(p, ng, np.int32), want.ravel())
    r = d.download_grains()
    assert r["cell"].size == n
    if n:
        env = host(e, (n, 4), np.float64)
        assert np.array_equal(env, r["env"])
        assert np.array_equal(f["gid"].ravel()[r["cell"]], np.arange(n))
        assert np.array_equal(f["ori"].ravel()[r["cell"]], r["orient"])
        assert np.array_equal(f["env"].reshape(-1, 4)[r["cell"]], env)
    s.close()
