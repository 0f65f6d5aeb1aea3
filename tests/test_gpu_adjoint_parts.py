"""The F32C adjoint at sizes around its chunks and on both sides of the launch
rule that gives each phase of a super-tile pair its own block (up to 1,024
pairs: 8,192 particles), against the oracle per unit of summation scale, to
the bounds of the adjoint tests (1e-5; sigma 1e-4)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 65, 255, 257, 700, 8192, 8193])
@pytest.mark.parametrize("jbar", [True, False])
def test_sizes(vpm, orc, n, jbar):
    P = vpm.workloads.random_cloud(n, seed=n)
    P[:, 6] *= 2.0
    w, W = vpm.workloads.adjoint_weights(n, seed=n)
    if not jbar:
        W = np.zeros((n, 9))
    kernel = "gaussianerf" if n % 2 else "winckelmans"
    print(n, jbar, kernel, flush=True)
    got = vpm.uj_adjoint(P, w, W, kernel=kernel, precision="f32c")
    ref = orc.uj_adjoint(P, kernel, w, W)
    mag = orc.uj_adjoint_scale(P, kernel, w, W)
    for name, a, r, m, tol in zip(("X", "Gamma", "sigma"), got, ref, mag, (1e-5, 1e-5, 1e-4)):
        a, r, m = (np.asarray(x).reshape(n, -1) for x in (a, r, m))
        den = np.linalg.norm(m, axis=1)
        e = (np.linalg.norm(a - r, axis=1) / np.maximum(den, 1e-6 * den.max())).max()
        print("  ", name, "%.1e" % e, flush=True)
        assert np.all(np.isfinite(a)) and e < tol, (name, e)
