"""A refused allocation is reported once: it leaves no error behind for the
launches that follow it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_refused_allocation_leaves_no_error(vpm):
    P = vpm.workloads.random_cloud(300, seed=1)
    f = vpm.Field(300)
    f.set_particles(P)
    with pytest.raises(vpm.VPMError) as e:
        vpm.Field(2 ** 31 - 1)                 # 790 GB of particles
    assert e.value.status == vpm._lib.VPM_ENOMEM
    f.uj_direct("gaussianerf", "f32c")
    out = np.zeros_like(P)
    f.get_particles(out)
    f.close()
    assert np.all(np.isfinite(out)) and np.any(out[:, 9:12] != 0)
