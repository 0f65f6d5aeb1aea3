"""Entry points that write into the caller's particle matrix refuse a read-only
one (a view marked so, a file mapped for reading) before any work; those that
only read it take it."""
import numpy as np
import pytest


class _Library:
    """Stands in for the native library: every call succeeds and is counted."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return 0
        return call


@pytest.fixture
def native(vpm, monkeypatch):
    L = _Library()
    monkeypatch.setattr(vpm.api, "lib", lambda: L)
    monkeypatch.setattr(vpm.api, "_field_cache", {})
    return L


def _matrix(vpm, tmp_path, how):
    P = vpm.workloads.random_cloud(64, seed=2)
    if how == "view":
        P.flags.writeable = False
        return P
    np.save(tmp_path / "p.npy", P)
    return np.load(tmp_path / "p.npy", mmap_mode="r")


def _calls(vpm):
    api, z = vpm.api, ([0], [64], [0], [64])
    return {
        "UJ_hip": lambda P: api.UJ_hip(P),
        "UJ_hip sfs": lambda P: api.UJ_hip(P, reset_sfs=True, sfs=True),
        "UJ_hip_fields": lambda P: api.UJ_hip_fields(P.copy(), P),
        "p2p_ranges": lambda P: api.p2p_ranges(P, *z),
        "estr_ranges": lambda P: api.estr_ranges(P, *z),
        "zeta_ranges": lambda P: api.zeta_ranges(P, *z),
        "Estr_hip": lambda P: api.Estr_hip(P),
        "get_particles": lambda P: api.Field.get_particles(object.__new__(api.Field), P),
        "get_particles rows": lambda P: api.Field.get_particles(object.__new__(api.Field), P, rows=(9, 12)),
    }


@pytest.mark.parametrize("how", ["view", "mapped file"])
@pytest.mark.parametrize("name", ["UJ_hip", "UJ_hip sfs", "UJ_hip_fields", "p2p_ranges", "estr_ranges", "zeta_ranges",
                                  "Estr_hip", "get_particles", "get_particles rows"])
def test_refused_before_any_work(vpm, native, tmp_path, name, how):
    P = _matrix(vpm, tmp_path, how)
    before = P.copy()
    with pytest.raises(ValueError, match="read-only"):
        _calls(vpm)[name](P)
    assert native.calls == []
    assert np.array_equal(P, before)


def test_particle_field(vpm, native):
    pf = vpm.ParticleField(64)
    vpm.add_particles(pf, vpm.workloads.random_cloud(64, seed=2))
    pf.particles.flags.writeable = False
    with pytest.raises(ValueError, match="read-only"):
        vpm.UJ_hip(pf)
    assert native.calls == []


def test_accepted(vpm, native, tmp_path):
    P = _matrix(vpm, tmp_path, "mapped file")
    T = P.copy()
    vpm.UJ_hip_fields(P, T)                                    # a source is only read
    vpm.UJ_hip(T)
    vpm.UJ_hip(P[:0])                                          # nothing to write
    assert "vpm_uj_direct_fields" in native.calls and "vpm_uj_direct" in native.calls
