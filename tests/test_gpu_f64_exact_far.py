"""FP64 reference arithmetic: the pairs whose g and dg/dr (U/J) or zeta
(E_str) are 1, 0 and 0 to the last bit, which the all-pairs kernels evaluate
without them or skip."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _spread(n, q_at, seed):
    """n particles at distances from 1e-3 to 1e3 core sizes, some of them at
    q_at (just inside and outside) from the first, one coincident pair."""
    rng = np.random.default_rng(seed)
    e = rng.normal(size=(n, 3))
    e /= np.linalg.norm(e, axis=1)[:, None]
    X = e * 0.01 * 10 ** rng.uniform(-3, 3, (n, 1))
    X[0] = 0.0
    for k, q in enumerate((q_at * (1 - 1e-9), q_at * (1 + 1e-9), q_at * 1.001, q_at * 3)):
        X[2 + k] = q * 0.01 * e[2 + k]
    X[n - 1] = X[1]
    return X, rng.normal(size=(n, 3)), np.where(np.arange(n) % 3 == 2, 0.01 * rng.uniform(0.5, 2, n), 0.01)


def _estr(vpm, P, kernel):
    f = vpm.Field(P.shape[0])
    f.set_particles(P)
    f.estr_direct(kernel, "f64")
    out = P.copy()
    f.get_particles(out)
    return out


def _hold(A, R, scale):
    """Per unit of summation scale; e^-x is good to x ulps (x < 746), and
    subnormal zetas to one of theirs."""
    d = np.abs(A[:, 39:42] - R[:, 39:42]).max(axis=1)
    assert np.all(d <= 1e-12 * scale + 1e-290), (d / np.maximum(scale, 1e-290)).max()


@pytest.mark.parametrize("kernel,q", [("gaussianerf", 10.0), ("gaussian", 13 ** 0.5), ("winckelmans", 10.0),
                                      ("singular", 10.0)])
@pytest.mark.parametrize("n", [64, 65, 256])
def test_uj_bits(vpm, kernel, q, n):
    """One source with strength at a time, so that no order of summation
    matters: the all-pairs kernel has the bits of the list kernel, which
    evaluates g and dg/dr of every pair."""
    X, G, S = _spread(n, q, n)
    for case in ("plain", "sigma out of range", "great strength", "great distance"):
        P = vpm.fields.make_particles(X, G, S)
        if case == "sigma out of range":
            P[n // 2, 6] = 1e-120
        elif case == "great strength":
            P[n // 2, 3] = 1e300
        elif case == "great distance":
            P[n // 2, 1] = 1e120
        for j in (0, 1, 2, 3, 5, n // 2, n - 1):
            A = P.copy()
            A[:, 3:6] = 0.0
            A[j, 3:6] = P[j, 3:6]
            B = A.copy()
            print(kernel, n, case, j, flush=True)
            vpm.UJ_hip(A, kernel=kernel, precision="f64")
            vpm.p2p_ranges(B, [0], [n], [0], [n], kernel=kernel, precision="f64")
            assert np.array_equal(A[:, 9:24], B[:, 9:24], equal_nan=True), (case, j)
            assert case != "plain" or np.all(np.isfinite(A[:, 9:24]))


@pytest.mark.parametrize("kernel,q", [("gaussianerf", 39.0), ("gaussian", 83 ** 0.5), ("winckelmans", 39.0),
                                      ("singular", 1.0)])
@pytest.mark.parametrize("n", [65, 257])
def test_estr_skipped_sources(vpm, orc, kernel, q, n):
    """Against the oracle on the same U/J, per unit of summation scale; a NaN
    or infinite J far from every target still reaches every target."""
    X, G, S = _spread(n, q, n + 1)
    X[n // 2] = (1e3, 0.0, 0.0)      # past the cut of everything
    P = vpm.fields.make_particles(X, G, S)
    vpm.UJ_hip(P, kernel=kernel, precision="f64")
    A, R = _estr(vpm, P, kernel), P.copy()
    orc.estr_direct(R, kernel)
    _hold(A, R, orc.estr_scale(P, kernel))
    for bad in (np.nan, np.inf):
        B = P.copy()
        B[n // 2, 15:24] = bad
        print(kernel, n, bad, flush=True)
        assert not np.any(np.isfinite(_estr(vpm, B, kernel)[:, 39:42]))
