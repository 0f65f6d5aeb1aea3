"""The spatial sort on both sides of the size where counting gives way to the
radix sort, with coincident particles (equal keys): the zeta field of every
particle against the FP64 kernel, which runs in storage order.  All strengths
are positive, so no sum cancels and FP32 pairs keep 1e-5 (64 x 6e-8 for the
terms, exp2's argument included, and chains of 256)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 255, 257, 4096, 4097, 8192, 8193])
def test_sorted_zeta(vpm, n):
    rng = np.random.default_rng(n)
    P = vpm.workloads.random_cloud(n, seed=n)
    P[:, 3:6] = rng.uniform(0.5, 1.0, (n, 3))
    P[:, 6] = rng.uniform(0.1, 0.2, n)
    P[n // 2:n // 2 + n // 4, 0:3] = P[0:n // 4, 0:3]
    f = vpm.Field(n)
    got = []
    for precision in ("f32c", "f64"):
        f.set_particles(P)
        f.zeta_direct("gaussianerf", precision)
        out = np.zeros_like(P)
        f.get_particles(out, rows=(15, 18))
        got.append(out[:, 15:18])
    f.close()
    assert np.all(got[1] > 0)
    assert np.abs(got[0] / got[1] - 1).max() < 1e-5
