"""Particle kernel at the edges of its wavefronts, its batches of field bodies
and its chunks: every particle equals, bit for bit, the oracle's trajectory of
the same particle carried as one more body of the field."""
import tempfile

import numpy as np
import pytest

from ephemeris_amd import generator as gen
from ephemeris_amd.particles import ParticleSet
from oracle import pyoracle as po
from tests.util import bits_equal

pytestmark = pytest.mark.gpu

DT = 86400.0


# field bodies: below one batch, whole batches, a remainder, the most that are kept, past it;
# particles: one, one short of a wavefront, one more, past a block of 256
@pytest.mark.parametrize("bodies,count", [(1, 1), (2, 63), (3, 64), (4, 65), (8, 257), (9, 2), (10, 66), (25, 65)])
def test_particles_at_edges_match_oracle(bodies, count):
    f9 = gen.make_field9(gen.make_full())
    spec = gen.make_small() if bodies > 9 else f9
    spec = gen.SystemSpec(list(spec.bodies)[:bodies], delta_t=DT)
    r, v = gen.make_particles(count, seed=bodies, field9=f9)
    print(f"\n[case] {bodies} field bodies, {count} particles, 3 steps", flush=True)
    ps = ParticleSet.from_config(gen.write_system(spec, tempfile.mkdtemp(), "Field"), r, v)
    dt = DT if bodies <= 9 else 300.0
    ps.integrate(dt, 3)
    pr, pv, _ = ps.download()
    for i in {0, count // 2, count - 1}:
        s = gen.SystemSpec(list(spec.bodies) + [gen.particle_body(r[i], v[i])], delta_t=dt)
        o = po.OSystem.load(gen.write_system(s, tempfile.mkdtemp(), "FieldP"), pool_at_load=False)
        o.integrate(dt, 3, pool=True)
        for got, q in ((pr[i], "r"), (pv[i], "v")):
            ref = np.array([[o.masses[f"{q}_{c}_hi"][bodies], o.masses[f"{q}_{c}_lo"][bodies]] for c in "xyz"]).ravel()
            assert bits_equal(got, ref), (i, q)

