"""Row downloads of many ring pieces while the rows change: each download goes
through the pieces of the one before it, and a piece is read on its event with
later ones in flight, so a read too early shows the rows of another download."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows of 24 / 216 bytes: 2 and 5 pieces of 1 MiB at 60,007, 17 of 2.7 MB at 200,003
@pytest.mark.parametrize("n,rows", [(60007, (0, 3)), (60007, (0, 9)), (200003, (0, 27))])
def test_changing_rows(vpm, n, rows):
    rng = np.random.default_rng(n)
    P = rng.normal(size=(n, 46))
    P[:, 6] = rng.uniform(0.1, 1.0, n)
    f = vpm.Field(n)
    out = np.zeros_like(P)
    for k in range(6):
        P[:, 0:3] += 1.0
        P[:, 9:27] -= 1.0
        f.set_particles(P)
        f.get_particles(out, rows=rows)
        assert np.array_equal(out[:, rows[0]:rows[1]], P[:, rows[0]:rows[1]]), k
    f.close()
