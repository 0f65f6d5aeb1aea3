"""Particle transfers: field sizes around one, three and four ring pieces
(2,849 records of 368 bytes each), around the sizes where uploads leave the
ring (5,698) and come back to it (91,180), whole records and
row ranges, rows outside a range left alone, the first bad record reported
from any worker's share, and nothing changed by a refused upload."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1425, 2849, 2850, 5698, 5699, 8547, 8548, 60007, 91180, 91181])
def test_round_trip(vpm, n):
    rng = np.random.default_rng(n)
    P = rng.normal(size=(n, 46))
    P[:, 6] = rng.uniform(0.1, 1.0, n)
    f = vpm.Field(n + 20000)
    f.set_particles(P)
    out = np.full_like(P, -1.0)
    f.get_particles(out)
    assert np.array_equal(out, P)
    for r0, r1 in ((0, 1), (6, 7), (9, 27), (39, 42), (1, 46)):
        out = np.full_like(P, -1.0)
        f.get_particles(out, rows=(r0, r1))
        assert np.array_equal(out[:, r0:r1], P[:, r0:r1])
        assert np.all(out[:, :r0] == -1.0) and np.all(out[:, r1:] == -1.0)
    m = (n + 1) // 2           # fewer than the field holds
    out = np.full_like(P, -1.0)
    f.get_particles(out, rows=(3, 6), np_=m)
    assert np.array_equal(out[:m, 3:6], P[:m, 3:6]) and np.all(out[m:] == -1.0)
    Q = P[: min(n, 15000)]     # appended after the others
    f.add_particles(Q)
    out = np.zeros((n + len(Q), 46))
    f.get_particles(out)
    assert np.array_equal(out[:n], P) and np.array_equal(out[n:], Q)
    f.close()


def test_bad_records(vpm):
    n = 100007
    P = vpm.workloads.random_cloud(n, seed=3)
    f = vpm.Field(2 * n)
    f.set_particles(P)
    for k, row, v, what in ((99999, 2, np.nan, "non-finite"), (31234, 6, 0.0, "sigma"), (17, 4, np.inf, "non-finite")):
        B = P.copy()
        B[k, row] = v
        B[n - 1, 6] = -1.0
        for call in (f.set_particles, f.add_particles):
            with pytest.raises(vpm.VPMError) as e:
                call(B)
            assert what in str(e.value) and ("particle %d" % k) in str(e.value)
        assert f.np == n
    out = np.zeros_like(P)
    f.get_particles(out)
    assert np.array_equal(out, P)
    f.close()
