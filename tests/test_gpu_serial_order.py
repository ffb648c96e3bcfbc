"""The single-thread-order main force with one workgroup per body
(k_main_serial_wpb) against the one-thread-per-body kernel, bit for bit: a
force evaluation at sizes around its 64-partner tiles and its rounds of four
tiles, with every model, and batches that take two and one wavefronts per
body; and an integration of small systems that now take the launches."""
import numpy as np
import pytest

from ephemeris_amd import _lib
from ephemeris_amd.layout import MASS_DTYPE
from ephemeris_amd.system import GpuSystems
from tests.util import GOLDEN, bits_equal, load_npz

pytestmark = pytest.mark.gpu


def _subset(n, copies=1):
    """The n most massive bodies of the 504-body system, `copies` times."""
    d = load_npz(GOLDEN / "accel_full504_pool.npz")
    m = d["masses_in"]
    m = m[np.sort(np.argsort(-m["GM"], kind="stable")[:n])]
    return np.concatenate([m] * copies), np.full(copies, n), d["gps"], d["rings"]


def _both(args, call):
    out = []
    for variant in (0, 1):
        g = GpuSystems(*args)
        g.set_variant(variant, allow_persistent=variant == 0)
        call(g)
        out.append(g.download()[0])
        g.close()
    return [f for f in MASS_DTYPE.names if not bits_equal(out[0][f], out[1][f])]


@pytest.mark.parametrize("n,copies", [(1, 1), (2, 1), (63, 1), (64, 1), (65, 1), (128, 1), (257, 1), (504, 1),
                                      (130, 9), (70, 40)])
def test_accel_equals_one_thread_per_body(n, copies):
    print(f"\n[case] serial-order accel, {copies} x {n} bodies", flush=True)
    assert not _both(_subset(n, copies), lambda g: g.accel(_lib.SUMMATION_SERIAL))


@pytest.mark.parametrize("n,copies", [(1, 1), (2, 1), (3, 1), (16, 1), (17, 1), (33, 1), (40, 3), (48, 1), (48, 60)])
@pytest.mark.parametrize("models,lag", [(True, True), (False, True), (False, False)])
def test_small_systems_integrate_alike(n, copies, models, lag):
    """On the path that the library chooses (the persistent workgroup or the
    launches), with and without models and time lags, against one thread per
    body; the sizes are the edges of its 16- and 48-body layouts."""
    print(f"\n[case] {copies} x {n} bodies, models {models}, time lags {lag}, 3 steps", flush=True)
    m, sys_n, gps, rings = _subset(n, copies)
    if not models:
        m["gp"], m["ring"] = -1, -1
    if not lag:
        m["tide_delay"] = 0.0
    assert not _both((m, sys_n, gps, rings), lambda g: g.integrate(300.0, 3))


def test_spin_at_rest_and_undefined():
    """Bodies without spin take one spin step instead of four, and a body
    whose GL is not finite has it set from its spin: the bits of one thread
    per body, persistent and in launches."""
    print("\n[case] 12 bodies, some at rest, one with GL undefined, 3 steps", flush=True)
    for models in (True, False):
        m, sys_n, gps, rings = _subset(12)
        for c in "xyz":
            m[f"w_{c}"][3:6] = 0.0
            for part in ("hi", "lo"):
                m[f"GL_{c}_{part}"][3:6] = 0.0
            m[f"GL_{c}_hi"][7] = np.nan
        if not models:
            m["gp"], m["ring"] = -1, -1
        assert not _both((m, sys_n, gps, rings), lambda g: (g.accel(), g.integrate(300.0, 3)))
