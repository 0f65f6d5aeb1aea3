"""One rule for the far kernel, whatever a call returns: U/J alone, U/J with
E_str, and U/J followed by E_str start from the same J, and E_str, a sum of
differences of J, is no less precise for it.  The figures are the RMS of the
error per unit of the summation scale with every pair of U/J in FP32 on these
fields; the far kernel's shorter chains leave less than three quarters."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _moved(P):
    rng = np.random.default_rng(3)
    step = P[:, 6].min() / 3
    P[:, 0:3] += rng.uniform(-0.1 * step, 0.1 * step, (len(P), 3))
    P[:, 3:6] *= 1 + 0.05 * rng.normal(size=(len(P), 1))
    return P


FIELDS = {
    "leapfrog": (lambda W: _moved(W.leapfrog_cfg2(Nphi=128)), 1.39e-6),
    "ring": (lambda W: _moved(W.ring_test(Nphi=16384, Rcross=12 * math.pi / 16384)), 5.33e-5),
    "jet": (lambda W: W.jet_column(16384, seed=1), 2.80e-5),
}


@pytest.mark.parametrize("name", sorted(FIELDS))
def test_estr_from_the_same_j(vpm, orc, name):
    make, figure = FIELDS[name]
    P = make(vpm.workloads)
    f = vpm.Field(len(P))
    f.set_particles(P)
    ref, alone, both, after = (np.zeros_like(P) for _ in range(4))
    f.uj_direct("gaussianerf", "f64", reset_sfs=True, sfs=True)
    f.get_particles(ref)
    f.uj_direct("gaussianerf", "f32c", reset_sfs=True)
    f.get_particles(alone)
    f.estr_direct("gaussianerf", "f32c")
    f.get_particles(after)
    f.uj_direct("gaussianerf", "f32c", reset_sfs=True, sfs=True)
    f.get_particles(both)
    f.close()
    assert np.array_equal(alone[:, 9:24], both[:, 9:24])
    s = orc.estr_scale(ref, "gaussianerf")
    for what, got in (("U/J with E_str", both), ("U/J, then E_str", after)):
        e = np.linalg.norm(got[:, 39:42] - ref[:, 39:42], axis=1) / s
        rms = math.sqrt((e * e).mean())
        print("%s %s rms %.2e max %.2e" % (name, what, rms, e.max()), flush=True)
        assert rms <= 0.75 * figure
