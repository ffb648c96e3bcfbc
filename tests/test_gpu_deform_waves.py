"""The deformation with two and four wavefronts per body, two partners per
lane, against one wavefront per body and one thread per body, bit for bit:
sizes around its 64-partner chunks, its rounds of 256 and 512 partners (257
bodies on two wavefronts take two rounds and re-form the pairs in each spin
pass), bodies with and without time lags, and a spin at rest, where the tidal
axis of the partners is taken in the language's operations."""
import numpy as np
import pytest

from ephemeris_amd.layout import MASS_DTYPE
from ephemeris_amd.system import GpuSystems
from tests.util import GOLDEN, bits_equal, load_npz

pytestmark = pytest.mark.gpu

CASES = [(1, 12), (1, 63), (1, 65), (1, 127), (1, 128), (1, 129), (1, 255), (1, 257), (1, 504), (5, 50), (9, 60)]


@pytest.mark.parametrize("copies,n", CASES)
@pytest.mark.parametrize("kind", ["as is", "all lag", "at rest"])
def test_bits(copies, n, kind):
    print(f"\n[case] {copies} x {n} bodies, {kind}: accel and 2 steps", flush=True)
    d = load_npz(GOLDEN / "accel_full504_pool.npz")
    m = d["masses_in"]
    m = m[np.sort(np.argsort(-m["GM"], kind="stable")[:n])]
    if kind == "all lag":
        m["k2"], m["k2r"], m["tide_delay"] = 0.3, 0.3, 600.0
    elif kind == "at rest":
        for c in "xyz":
            m[f"w_{c}"][::2] = 0.0
            for part in ("hi", "lo"):
                m[f"GL_{c}_{part}"][::2] = 0.0
                m[f"v_{c}_{part}"][:] = 0.0
    args = np.concatenate([m] * copies), np.full(copies, n), d["gps"], d["rings"]
    out = []
    for variant, waves in ((1, 0), (2, 1), (2, 2), (2, 4)):
        g = GpuSystems(*args)
        g.set_variant(variant, allow_persistent=False)
        g.set_waves(waves)
        g.accel()
        a = g.download()[0]
        g.integrate(300.0, 2)
        out.append((a, g.download()[0]))
        g.close()
    for i, what in enumerate(("accel", "integrate")):
        for o in out[1:]:
            bad = [f for f in MASS_DTYPE.names if not bits_equal(out[0][i][f], o[i][f])]
            assert not bad, f"{what}: {bad}"
