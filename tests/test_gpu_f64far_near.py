"""The FP64 far-form path's Gaussian-erf near pair (FP64 fits of the reduced
kernel functions) against mpmath, one pair at a time."""
import mpmath as mp
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(d, G, sigma):
    """U and J (J[3 b + a] = du_a/dx_b) at separation d of one source, 40 digits."""
    with mp.workdps(40):
        d, G = [mp.mpf(float(x)) for x in d], [mp.mpf(float(x)) for x in G]
        r2 = sum(x * x for x in d)
        r = mp.sqrt(r2)
        q = r / mp.mpf(sigma)
        qdg = mp.sqrt(2 / mp.pi) * q ** 3 * mp.exp(-q * q / 2)
        g = mp.erf(q / mp.sqrt(2)) - qdg / q ** 2
        w = -1 / (4 * mp.pi * r2 * r)
        c = [w * (d[1] * G[2] - d[2] * G[1]), w * (d[2] * G[0] - d[0] * G[2]), w * (d[0] * G[1] - d[1] * G[0])]
        J = [[(qdg - 3 * g) / r2 * c[a] * d[b] for a in range(3)] for b in range(3)]
        W = [g * w * x for x in G]
        for b, a, v in ((0, 1, -W[2]), (0, 2, W[1]), (1, 0, W[2]), (1, 2, -W[0]), (2, 0, -W[1]), (2, 1, W[0])):
            J[b][a] += v
        return np.array([float(g * x) for x in c]), np.array([float(x) for row in J for x in row])


@pytest.mark.parametrize("q", [1e-6, 1e-3, 0.1, 1.0, 2 * (1 - 1e-12), 2 * (1 + 1e-12), 3.0, 5.0, 9.9, 10.1, 30.0, 1e3])
def test_near_pair_vs_mpmath(vpm, q):
    """Both particles lie in their wave's target box, so the pair takes the
    near form at every q.  Each of F' and H'' is good to about ten roundings,
    and J's terms are no larger than three times J: 1e-14 (45 ulps)."""
    sigma = 0.03
    e = np.array([0.3, -0.7, 0.5])
    X = np.vstack([np.zeros(3), q * sigma * e / np.linalg.norm(e)])
    G = np.array([[0.4, -1.1, 0.7], [0.0, 0.0, 0.0]])
    P = vpm.fields.make_particles(X, G, np.full(2, sigma))
    vpm.UJ_hip(P, kernel="gaussianerf", precision="f64far")
    U, J = _pair(X[1] - X[0], G[0], sigma)
    eu = np.linalg.norm(P[1, 9:12] - U) / np.linalg.norm(U)
    ej = np.linalg.norm(P[1, 15:24] - J) / np.linalg.norm(J)
    print("q %.13g U %.1e J %.1e" % (q, eu, ej), flush=True)
    assert eu < 1e-14 and ej < 1e-14
