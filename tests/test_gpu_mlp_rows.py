"""The fused inference kernel with unscaled activations (every call on rows of
the network except amca_mlp_forward_fused) against the CPU oracle at the edges
of its 64-row groups, of one group per CU and of eight per work-group, through
the host-row and the device-row entry points, and after each way of changing
the parameters."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as mo  # noqa: E402
from test_gpu_mlp import _params  # noqa: E402
from test_zz_no_alloc import _Hip  # noqa: E402

pytestmark = pytest.mark.gpu


def _check(t, p, X):
    ref, _ = mo.forward(p.astype(np.float64), X)
    s = np.abs(ref).max() + 1
    # same rounding points: the FP32 accumulation order, and now and then an
    # activation on the other side of a BF16 rounding boundary (2^-9 of it)
    np.testing.assert_allclose(t, ref, rtol=0, atol=2e-2 * s)
    assert np.median(np.abs(t - ref)) < 1e-5 * s


@pytest.mark.parametrize("n", [1, 32, 33, 64, 65, 127, 256 * 64, 256 * 64 + 1, 8 * 256 * 64 + 65])
def test_rows_match_oracle(amca, n):
    from amca3d_amd import surrogate as S
    m = S.MLP(1)
    p = _params(9)
    m.set_params(p)
    X = np.random.default_rng(n).uniform(-1, 1, (n, 5)).astype(np.float32)
    t = m.forward(X)
    _check(t, p, X)
    hip = _Hip()
    guard = 64
    dX, dT = hip.upload(X), hip.upload(np.full(n + guard, np.nan, np.float32))
    assert S.lib().amca_mlp_forward_device(m.h, n, dX, dT) == 0
    got = hip.download(dT, np.empty(n + guard, np.float32))
    np.testing.assert_array_equal(got[:n].view(np.uint32), t.view(np.uint32))
    assert np.isnan(got[n:]).all()  # nothing past the last row
    hip.close()
    m.close()


def test_rows_follow_the_parameters(amca):
    from amca3d_amd import surrogate as S
    rng = np.random.default_rng(3)
    X = rng.uniform(-1, 1, (500, 5)).astype(np.float32)
    m = S.MLP(4)  # as created
    _check(m.forward(X), m.params(), X)
    m.set_params(_params(11))
    _check(m.forward(X), m.params(), X)
    hip = _Hip()
    Y = rng.uniform(-1, 1, 500).astype(np.float32)
    before = m.params()
    dX, dY = hip.upload(X), hip.upload(Y)
    assert S.lib().amca_mlp_train_device(m.h, 500, dX, dY, 250, 7, 1e-3, 5, None) == 0
    assert not np.array_equal(before, m.params())
    _check(m.forward(X), m.params(), X)
    hip.close()
    m.close()
