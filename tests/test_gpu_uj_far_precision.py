"""Precision of the F32C far field on the matrix cores (the sums of
test_gpu_uj_far.py are bounded there; here they are held to their precision).

Whole fields: the error of U and J per unit of the scale of their sums,
s = sum |term|, is no larger than with every pair in FP32 (the figures are
those of the FP32 pair kernel on these fields, before there was a far kernel),
and each target stays within 1e-6 of its scale: FP32 chains of 64 near pairs
carry 64^(1/2) half-roundings, 2.4e-7, and four times that is allowed.

Single pairs: with one source of nonzero strength each target has one term,
and nothing averages.  In roundings of 2^-24: positions of three components at
r = R / 8 leave 42 in r^2, truncated products 20, its sums 20, so 2.5 x 82 =
205 in r^-5; rsq, products and the FP16 halves of r^-5 27; the polynomials'
terms reach 27 r^3 for U at |s| = 2 r, and columns, chain and the product of
low halves add (4 + 6 + 4) x 27 = 378: 610 x 2^-24 = 3.6e-5 at the worst, and a
sixth of that in the mean square over the targets.  A lost half is 1.4e-4."""
import math

import numpy as np
import pytest
from test_gpu_uj_far import _exact

pytestmark = pytest.mark.gpu


def _leapfrog(W):
    P = W.leapfrog_cfg2(Nphi=512)
    rng = np.random.default_rng(3)
    step = P[:, 6].min() / 3
    P[:, 0:3] += rng.uniform(-0.1 * step, 0.1 * step, (len(P), 3))
    P[:, 3:6] *= 1 + 0.05 * rng.normal(size=(len(P), 1))
    return P


@pytest.mark.parametrize("name,make,u,j", [
    ("jet", lambda W: W.jet_column(262144, seed=1), 1.56e-8, 5.07e-8),
    ("leapfrog", _leapfrog, 1.65e-8, 7.67e-8),
    ("cloud", lambda W: W.random_cloud(65536, seed=1), 1.95e-9, 8.15e-9),
])
def test_no_worse_than_fp32_pairs(vpm, name, make, u, j):
    P = make(vpm.workloads)
    n = len(P)
    out = P.copy()
    vpm.UJ_hip(out, kernel="gaussianerf", precision="f32c")
    e = []
    for i in np.linspace(0, n - 1, 300).astype(int):
        U, J, su, sj = _exact("gaussianerf", P, P[i, 0:3])
        e.append((np.linalg.norm(out[i, 9:12] - U) / su, np.linalg.norm(out[i, 15:24] - J) / sj))
    e = np.array(e)
    rms = np.sqrt((e * e).mean(axis=0))
    print("%s U rms %.2e max %.2e J rms %.2e max %.2e" % (name, rms[0], e[:, 0].max(), rms[1], e[:, 1].max()), flush=True)
    # 300 targets: the mean square is known to 4 %
    assert rms[0] <= 1.04 * u and rms[1] <= 1.04 * j
    assert e.max() <= 1e-6


@pytest.mark.parametrize("field", ["cloud", "jet"])
@pytest.mark.parametrize("at", [0, 7000, 16420])
def test_single_pairs(vpm, field, at):
    n = 16421
    P = vpm.workloads.random_cloud(n, seed=4) if field == "cloud" else vpm.workloads.jet_column(n, seed=4)
    G = P[at, 3:6].copy()
    P[:, 3:6] = 0.0
    P[at, 3:6] = G
    out = P.copy()
    vpm.UJ_hip(out, kernel="gaussianerf", precision="f32c")
    keep = np.arange(n) != at
    d, sigma = (P[:, 0:3] - P[at, 0:3])[keep], P[at, 6]
    r = np.linalg.norm(d, axis=1)
    q = r / sigma
    a = math.sqrt(2 / math.pi) * q * np.exp(-0.5 * q * q)
    g = np.array([math.erf(min(x, 30.0) / math.sqrt(2)) for x in q]) - a
    F, H = g / r ** 3, (a * q * q - 3 * g) / r ** 5
    Gp = -G / (4 * np.pi)
    v = np.cross(d, Gp)
    U = F[:, None] * v
    J = (H[:, None, None] * d[:, :, None] * v[:, None, :]).reshape(-1, 9)      # J[3 b + a] = v_a d_b
    W = F[:, None] * Gp
    z = np.zeros(n - 1)
    J += np.stack([z, -W[:, 2], W[:, 1], W[:, 2], z, -W[:, 0], -W[:, 1], W[:, 0], z], 1)
    m = np.linalg.norm(Gp)
    eu = np.linalg.norm(out[keep, 9:12] - U, axis=1) / (F * r * m)
    ej = np.linalg.norm(out[keep, 15:24] - J, axis=1) / ((np.abs(H) * r * r + F) * m)
    for what, e in (("U", eu), ("J", ej)):
        rms = math.sqrt((e * e).mean())
        print("%s %d %s max %.2e rms %.2e" % (field, at, what, e.max(), rms), flush=True)
        assert e.max() <= 3.6e-5 and rms <= 6e-6
