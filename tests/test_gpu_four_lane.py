"""The four-lanes-per-body kernels (set_variant(4)) against the
one-thread-per-body kernels, bit for bit, in thread-pool order: sizes around
their 16-body blocks, 16-partner tiles and groups of four, with bodies whose
quadrupole, spin or luminosity is nowhere, everywhere, first or last (which
decides what rows of terms a group writes and adds), and bodies that carry
both a geopotential and a ring among the receivers."""
import numpy as np
import pytest

from ephemeris_amd import _lib
from ephemeris_amd.layout import MASS_DTYPE
from ephemeris_amd.system import GpuSystems
from tests.util import GOLDEN, bits_equal, load_npz

pytestmark = pytest.mark.gpu


def _systems(sizes, kind):
    d = load_npz(GOLDEN / "accel_full504_pool.npz")
    heavy = np.argsort(-d["masses_in"]["GM"], kind="stable")
    parts = []
    for n in sizes:
        idx = np.sort(heavy[:n])
        if kind == "last":
            idx = idx[::-1]
        elif kind == "plain":                             # no quadrupole, no light, no model
            idx = np.sort(heavy[-n:])
        m = d["masses_in"][idx].copy()
        if kind == "all":                                 # every body has a quadrupole and shines
            m["C_static_xx"], m["C_static_zz"], m["lum"], m["recpt"] = 1e-4, -1e-4, 1e20, 1.0
            m["rR2G_4c"] = 1e-12
        elif kind == "plain":
            m["gp"], m["ring"] = -1, -1
            for f in MASS_DTYPE.names:
                if f.startswith("C_static") or f in ("lum", "k2", "k2r", "tide_delay"):
                    m[f] = 0
        parts.append(m)
    return np.concatenate(parts), np.array(sizes), d["gps"], d["rings"]


@pytest.mark.parametrize("kind", ["first", "last", "all", "plain"])
@pytest.mark.parametrize("sizes", [(49,), (63, 64, 65), (80, 81, 95, 96, 97), (127, 50, 129), (504, 52, 255)])
def test_equals_one_thread_per_body(sizes, kind):
    print(f"\n[case] sizes {sizes}, {kind}: accel and 2 steps", flush=True)
    args = _systems(sizes, kind)
    out = []
    for variant in (4, 1):
        g = GpuSystems(*args)
        g.set_variant(variant, allow_persistent=False)
        g.accel(_lib.SUMMATION_POOL)
        a = g.download()[0]
        g.integrate(300.0, 2)
        out.append((a, g.download()[0]))
        g.close()
    for i, what in enumerate(("accel", "integrate")):
        bad = [f for f in MASS_DTYPE.names if not bits_equal(out[0][i][f], out[1][i][f])]
        assert not bad, f"{what}: {bad}"
