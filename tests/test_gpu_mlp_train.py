"""The two training kernels against the CPU oracle at the edges of their 64-row
groups and of one group per work-group (256 of them: larger batches take several
groups each), their repeatability, and the loss trace across the stretch of
losses kept on the device."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as mo  # noqa: E402
from test_gpu_mlp import _params  # noqa: E402
from test_zz_no_alloc import _Hip  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 256 * 64 - 1, 256 * 64 + 1, 2 * 256 * 64 + 65])
def test_gradients_match_oracle(amca, n):
    from amca3d_amd.surrogate import MLP
    m = MLP(1)
    p = _params(13)
    m.set_params(p)
    rng = np.random.default_rng(n)
    X = rng.uniform(-1, 1, (n, 5)).astype(np.float32)
    Y = rng.uniform(-1, 1, n).astype(np.float32)
    g, loss = m.gradients(X, Y)
    again, loss2 = m.gradients(X, Y)
    np.testing.assert_array_equal(g.view(np.uint32), again.view(np.uint32))  # sums in a fixed order
    assert loss == loss2
    ref, rloss = mo.gradients(p.astype(np.float64), X, Y)
    assert loss == pytest.approx(rloss, rel=1e-3)
    off, _ = mo.layout()
    # same rounding points except dW5, whose dT the kernel keeps in FP32 (BF16 in
    # the oracle: 2^-9 relative per row): the oracle test's bound
    for l, ((w, b), fo) in enumerate(zip(off, mo.FAN_OUT)):
        for lo, hi, what in ((w, b, "W"), (b, b + fo, "b")):
            err = np.linalg.norm(g[lo:hi] - ref[lo:hi])
            assert err <= 2e-2 * np.linalg.norm(ref[lo:hi]) + 1e-7, (l, what, err)
    g64, _ = mo.gradients64(p.astype(np.float64), X, Y)
    assert np.linalg.norm(g - g64) < 5e-2 * np.linalg.norm(g64)
    m.close()


def test_adam_steps_and_loss_trace(amca):
    """Steps on one batch against Adam on the library's own gradients, and a
    trace longer than the losses kept on the device (4096 steps)."""
    from amca3d_amd import surrogate as S
    rng = np.random.default_rng(2)
    n = 130
    X = rng.uniform(-1, 1, (n, 5)).astype(np.float32)
    Y = rng.uniform(-1, 1, n).astype(np.float32)
    hip = _Hip()
    dX, dY = hip.upload(X), hip.upload(Y)
    m, ref = S.MLP(1), S.MLP(1)
    p0 = _params(17)
    m.set_params(p0)
    steps = 4100
    trace = np.full(steps, np.nan, np.float32)
    st = S.lib().amca_mlp_train_device(m.h, n, dX, dY, n, 6, 1e-3, 9, S._p(trace))
    assert st == 0
    p = p0.astype(np.float64)
    mm, vv = np.zeros_like(p), np.zeros_like(p)
    for it in range(6):
        ref.set_params(p.astype(np.float32))
        g, loss = ref.gradients(X, Y)
        # the two parameter vectors differ by FP32 rounding: of 50 433 weights about 50 lie
        # so near a BF16 boundary (2^-24 against a spacing of 2^-8) that they round the
        # other way, each moving a pre-activation by 2^-8 of one of its 128 terms and the
        # loss by parts in 1e5
        assert trace[it] == pytest.approx(loss, rel=2e-4)
        mm = 0.9 * mm + 0.1 * g
        vv = 0.999 * vv + 0.001 * g.astype(np.float64) ** 2
        p -= 1e-3 * (mm / (1 - 0.9 ** (it + 1))) / (np.sqrt(vv / (1 - 0.999 ** (it + 1))) + 1e-8)
    # FP32 moments and updates against 64 bits: 2^-24 of a weight each step, and where a
    # gradient is near zero a step of its own sign's uncertainty (at most 2 lr a step)
    d = np.abs(m.params() - p)
    assert np.median(d) < 1e-6 and np.quantile(d, 0.999) < 1e-4 and d.max() <= 6 * 2e-3
    # steps so small that neighbouring losses agree (each moves a weight by at most about
    # lr = 1e-7, the loss of 0.2 by parts in 1e5; a fitted network's loss would wander
    # by tens of percent a step): the trace is continuous where its stretches meet
    m.set_params(p0)
    trace[:] = np.nan
    st = S.lib().amca_mlp_train_device(m.h, n, dX, dY, n, steps, 1e-7, 9, S._p(trace))
    assert st == 0
    assert np.isfinite(trace).all() and trace[-1] < trace[0]
    assert np.abs(np.diff(trace.astype(np.float64)) / trace[:-1]).max() < 2e-3
    _, loss = m.gradients(X, Y)  # one step past the last traced loss
    assert loss == pytest.approx(trace[-1], rel=2e-3)
    hip.close()
    m.close()
    ref.close()


def test_training_right_after_create_repeats(amca):
    """A network's first steps use the parameters it was created with (its setup is
    complete when create or set_params returns), so two of a seed end the same."""
    from amca3d_amd import surrogate as S
    rng = np.random.default_rng(8)
    X = rng.uniform(-1, 1, (256, 5)).astype(np.float32)
    Y = rng.uniform(-1, 1, 256).astype(np.float32)
    hip = _Hip()
    dX, dY = hip.upload(X), hip.upload(Y)
    first = None
    for _ in range(20):
        m = S.MLP(5)
        assert S.lib().amca_mlp_train_device(m.h, 256, dX, dY, 256, 3, 1e-3, 9, None) == 0
        p = m.params()
        m.close()
        first = p if first is None else first
        np.testing.assert_array_equal(p.view(np.uint32), first.view(np.uint32))
    hip.close()


def test_set_params_starts_training_anew(amca):
    """Setting the parameters also sets Adam's moments to zero, every one of them: steps
    after other steps end as the first ones did."""
    from amca3d_amd import surrogate as S
    rng = np.random.default_rng(9)
    X = rng.uniform(-1, 1, (64, 5)).astype(np.float32)
    Y = rng.uniform(-1, 1, 64).astype(np.float32)
    hip = _Hip()
    dX, dY = hip.upload(X), hip.upload(Y)
    m = S.MLP(5)
    ends = []
    for lr in (1e-3, 3e-2, 1e-3):
        m.set_params(_params(4))
        assert S.lib().amca_mlp_train_device(m.h, 64, dX, dY, 64, 5, lr, 9, None) == 0
        ends.append(m.params().view(np.uint32))
    np.testing.assert_array_equal(ends[0], ends[2])
    assert (ends[0] != ends[1]).mean() > 0.9
    hip.close()
    m.close()
