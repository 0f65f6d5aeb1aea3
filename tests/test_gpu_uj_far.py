"""F32C all-pairs U/J with the far field on the matrix cores (taken from 2^28
pairs): sampled targets against FP64 sums, over fields that reach its edges --
the smallest size of its range, ragged sizes, target and source counts that
differ, coincident particles, strengths spread over
twelve decades with whole tiles of zeros, and domains of 1e-4 and 1e5.

Each target is held to the scale of its sums, s_i = sum |term|: 1e-5 s_i for U
and J.  A pair's FP32 coefficient carries at most ~20 roundings (r^-5 from r^2
turns one into 2.5), its expansion about the block origin loses at most 3 bits
at |s| = 2 r, and FP32 chains are at most 64 pairs (near) or one 256-source
tile (far): below 160 x 6e-8."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K4 = 1 / (4 * np.pi)


def _erf(x):
    import math
    return np.vectorize(math.erf)(x)


def _exact(kernel, S, x):
    """U (3,), J (9,), and the scales of their sums at target x in FP64."""
    d = x - S[:, 0:3]
    r2 = (d * d).sum(1)
    keep = r2 > 0
    d, r2, G, sg = d[keep], r2[keep], S[keep, 3:6], S[keep, 6]
    r = np.sqrt(r2)
    q = r / sg
    if kernel == "gaussian":
        g, k = -np.expm1(-q ** 3), 3 * q ** 3 * np.exp(-q ** 3)
    else:
        far = q > 12
        e = np.where(far, 1.0, 0.0)
        e[~far] = _erf(q[~far] / np.sqrt(2)) if (~far).any() else 0.0
        a = np.sqrt(2 / np.pi) * q * np.exp(-0.5 * q * q)
        g, k = e - a, a * q * q
    F, H = g / r ** 3, (k - 3 * g) / r ** 5
    v = np.cross(d, -K4 * G)
    U = (F[:, None] * v).sum(0)
    J = np.einsum("j,ja,jb->ba", H, v, d)
    W = (F[:, None] * (-K4 * G)).sum(0)
    J = J + np.array([[0, -W[2], W[1]], [W[2], 0, -W[0]], [-W[1], W[0], 0]])
    nv, nG = np.linalg.norm(v, axis=1), K4 * np.linalg.norm(G, axis=1)
    return U, J.reshape(9), (F * nv).sum(), (np.abs(H) * nv * r + F * nG).sum()


def _check(kernel, S, X, out, idx):
    for i in idx:
        U, J, su, sj = _exact(kernel, S, X[i, 0:3])
        assert np.abs(out[i, 9:12] - U).max() <= 1e-5 * su, (i, out[i, 9:12], U, su)
        assert np.abs(out[i, 15:24] - J).max() <= 1e-5 * sj, (i, out[i, 15:24], J, sj)


def _sample(n, rng):
    return np.unique(np.concatenate([[0, 1, n - 2, n - 1], rng.integers(0, n, 60)]))


def _spread(W, rng):
    P = W.random_cloud(17000, seed=5)
    P[:, 3:6] *= 10.0 ** rng.uniform(-12, 0, (17000, 1))
    P[P[:, 0] < 0.25, 3:6] = 0.0
    return P


def _twins(W, rng):
    P = W.jet_column(17001, seed=6)
    P[8000:9000, 0:3] = P[0:1000, 0:3]
    return P


def _apart(W, rng):
    P = W.random_cloud(16500, seed=7)
    P[::2, 0:3] += np.array([1000.0, -300.0, 0.0])
    return P


def _scaled(f):
    def make(W, rng):
        P = W.random_cloud(16421, seed=8)
        P[:, 0:3] = P[:, 0:3] * f + 3 * f
        P[:, 6] *= f
        return P
    return make


FIELDS = {
    "leapfrog_16384": lambda W, rng: W.leapfrog_cfg2(Nphi=128),
    "cloud_16421": lambda W, rng: W.random_cloud(16421, seed=4),
    "jet_20011": lambda W, rng: W.jet_column(20011, seed=4),
    "spread": _spread, "twins": _twins, "apart": _apart,
    "small_domain": _scaled(1e-4), "large_domain": _scaled(1e5),
}


@pytest.mark.parametrize("kernel", ["gaussianerf", "gaussian"])
@pytest.mark.parametrize("name", sorted(FIELDS))
def test_far_field(vpm, name, kernel):
    rng = np.random.default_rng(11)
    P = FIELDS[name](vpm.workloads, rng)
    out = P.copy()
    vpm.UJ_hip(out, kernel=kernel, precision="f32c")
    _check(kernel, P, P, out, _sample(len(P), rng))


@pytest.mark.parametrize("nt,ns", [(2048, 131072), (140001, 2113)])
def test_far_field_two_fields(vpm, nt, ns):
    rng = np.random.default_rng(13)
    S = vpm.workloads.jet_column(ns, seed=10)
    T = vpm.workloads.random_cloud(nt, seed=11)
    T[:, 0:3] -= 0.5
    out = T.copy()
    vpm.UJ_hip_fields(S, out, kernel="gaussianerf", precision="f32c")
    _check("gaussianerf", S, T, out, _sample(nt, rng))


def test_far_field_noalloc(vpm):
    """vpm_uj_direct_noalloc takes the split with the source splits that its
    array holds (fewer than vpm_uj_direct's here, so another summation order)."""
    api = vpm.api
    rng = np.random.default_rng(14)
    P = vpm.workloads.random_cloud(16421, seed=4)
    f = api.Field(len(P))
    f.set_particles(P)
    cfg = api.make_config("gaussianerf", "f32c", True)
    assert api.lib().vpm_uj_direct_noalloc(f.handle, C.byref(cfg), api._lib.UJ_RESET) == 0
    out = np.zeros_like(P)
    f.get_particles(out, rows=(9, 24))
    f.close()
    _check("gaussianerf", P, P, out, _sample(len(P), rng))
