"""A strength that overflows FP32 in a field large enough for the far kernel:
the components that it does not enter stay what they are (as in storage order,
where every pair takes the FP32 pair code), to the bound of
test_gpu_uj_far.py."""
import numpy as np
import pytest
from test_gpu_uj_far import _exact, _sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["gaussianerf", "gaussian"])
def test_infinite_strength(vpm, kernel):
    n = 16421
    P = vpm.workloads.random_cloud(n, seed=4)
    at = 5000
    P[:, 3:6] *= 1e7                   # the others above FP16's range, unless scaled
    P[at, 3:6] = (1e40, 0.0, 0.0)      # d x Gamma has no x component
    got = []
    for sort in (True, False):
        out = P.copy()
        vpm.UJ_hip(out, kernel=kernel, precision="f32c", sort=sort)
        got.append(out)
    for rows in (slice(9, 12), slice(15, 24)):
        assert np.array_equal(np.isfinite(got[0][:, rows]), np.isfinite(got[1][:, rows]))
    S = P.copy()
    S[at, 3:6] = 0.0
    for i in _sample(n, np.random.default_rng(1)):
        if i == at:
            continue
        U, _, su, _ = _exact(kernel, S, P[i, 0:3])
        assert abs(got[0][i, 9] - U[0]) <= 1e-5 * su
