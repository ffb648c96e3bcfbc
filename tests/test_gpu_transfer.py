"""Bodies and particles between the caller's records and the resident state:
an upload and a download return every byte that was sent (sizes around the
16-body blocks of the transposition), an upload that changes the tidal
classes between two captured steps is taken over, and a particle set gives
its initial state back."""
import numpy as np
import pytest

from ephemeris_amd import generator as gen
from ephemeris_amd.particles import ParticleSet
from ephemeris_amd.system import GpuSystems
from tests.util import GOLDEN, bits_equal, load_npz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 65, 504])
def test_upload_download_round_trip(n):
    print(f"\n[case] round trip of {n} bodies", flush=True)
    d = load_npz(GOLDEN / "accel_full504_pool.npz")
    a, b = d["masses_in"][:n].copy(), d["masses_out"][:n].copy()
    g = GpuSystems(a, None, d["gps"], d["rings"])
    assert bits_equal(g.download()[0], a)
    g.upload(b)
    assert bits_equal(g.download()[0], b)


def test_upload_with_other_tidal_classes():
    print("\n[case] upload that changes the tidal classes between integrations", flush=True)
    d = load_npz(GOLDEN / "accel_full504_pool.npz")
    a = d["masses_in"].copy()
    b = a.copy()
    b["tide_delay"] = 0.0
    args = (None, d["gps"], d["rings"])
    g, ref = GpuSystems(a, *args), GpuSystems(b, *args)
    for s in (g, ref):
        s.set_variant(4)
    g.integrate(300.0, 2)
    g.upload(b, np.zeros((1, 2)))
    for s in (g, ref):
        s.integrate(300.0, 2)
    assert bits_equal(g.download()[0], ref.download()[0])


def test_particles_give_their_initial_state_back():
    print("\n[case] 300 particles, initial state", flush=True)
    f9 = gen.make_field9(gen.make_full())
    d = load_npz(GOLDEN / "accel_small25_serial.npz")
    r, v = gen.make_particles(300, field9=f9)
    ps = ParticleSet(GpuSystems(d["masses_in"][:9], None, d["gps"], d["rings"]), r, v)
    pr, pv, _ = ps.download()
    assert bits_equal(pr[:, ::2], r) and bits_equal(pv[:, ::2], v)
    assert not pr[:, 1::2].any() and not pv[:, 1::2].any()
