"""Direct lists of few leaves with many source ranges each, which the F32C
wave kernels serve with several waves per leaf (U/J and E_str), against the
oracle.  Tolerances are those of the list tests of test_gpu_uj.py and
test_gpu_estr_ranges.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lists(n, leaf, per, step, seed):
    """Every `step`-th leaf of `leaf` particles against `per` of the leaves, a
    few of the source ranges empty."""
    rng = np.random.default_rng(seed)
    starts = np.arange(0, n, leaf)
    tb, te, sb, se = [], [], [], []
    for a in starts[::step]:
        for c in rng.permutation(starts)[:per]:
            tb.append(a)
            te.append(min(a + leaf, n))
            sb.append(c)
            se.append(c if rng.random() < 0.1 else min(c + leaf, n))
    return tb, te, sb, se


# at least 4 ranges to a wave of leaves over 16 particles, 8 of shorter ones
@pytest.mark.parametrize("leaf,per,step", [(50, 7, 1), (50, 16, 1), (64, 17, 2), (27, 40, 3), (16, 100, 5),
                                           (8, 150, 7), (5, 15, 1), (1, 150, 50)])
@pytest.mark.parametrize("kernel", ["gaussianerf", "gaussian", "winckelmans"])
def test_few_leaves(vpm, orc, kernel, leaf, per, step):
    n = 1200
    P = vpm.workloads.random_cloud(n, seed=61)
    P[:, 6] *= 3.0
    lists = _lists(n, leaf, per, step, leaf)
    A, R = P.copy(), P.copy()
    print(kernel, leaf, per, step, len(lists[0]), flush=True)
    vpm.p2p_ranges(A, *lists, kernel=kernel, precision="f32c")
    orc.direct_ranges(R, kernel, *lists)
    hit = np.zeros(n, bool)
    for a, b in zip(lists[0], lists[1]):
        hit[a:b] = True
    assert np.all(A[~hit, 9:24] == 0)
    u = np.maximum(orc.u_scale_ranges(P, kernel, *lists), 1e-300)
    eu = (np.linalg.norm(A[:, 9:12] - R[:, 9:12], axis=1) / u)[hit].max()
    ej = vpm.metrics.err_stats(A[hit][:, 15:24], R[hit][:, 15:24])["max"]
    print("U to its scale %.1e J %.1e" % (eu, ej), flush=True)
    assert eu < 1e-5 and ej < 1e-5

    rng = np.random.default_rng(5)
    P[:, 15:24] = rng.normal(0, 1, (n, 9))
    P[:, 39:42] = rng.normal(0, 1e-3, (n, 3))
    A, R = P.copy(), P.copy()
    vpm.api.estr_ranges(A, *lists, kernel=kernel, precision="f32c")
    orc.estr_ranges(R, kernel, *lists)
    assert np.array_equal(A[~hit], P[~hit])
    s = orc.estr_scale_ranges(P, kernel, *lists)
    e = np.linalg.norm(A[:, 39:42] - R[:, 39:42], axis=1)
    assert (e / np.maximum(s, 1e-6 * s.max())).max() < 5e-5
