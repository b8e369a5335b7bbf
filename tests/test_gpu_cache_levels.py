"""GPU check of the half steps' cache hints, chosen by what a step moves (the state and the streamed
coefficients together within 288 MiB; the state alone; neither).  The hints change no value: around the
source of one random medium, cut out at three sizes, the runs are equal bit for bit until the wave can
have been at the smallest cut's boundary and back (at most 4 cells a step each way)."""
import numpy as np
import pytest

from biot_amd import Solver, media, ricker

pytestmark = pytest.mark.gpu

SMALL, NT = 64, 14


@pytest.mark.parametrize("precision,sides", [("fp32", (136, 184)), ("fp64", (112, 148)), ("fp16", (172, 232)),
                                             ("fp16c", (140,))])
def test_runs_do_not_depend_on_the_size_around_them(precision, sides):
    core = np.random.default_rng(4).uniform(0.95, 1.05, (SMALL,) * 3)
    core[30:34, 30:34, 30:34] = 1.1  # the largest moduli, and with them the storage scales, near the source
    core[26:30, 26:30, 26:30] = 0.9
    ref = None
    for side in (SMALL,) + sides:
        print(f"cache levels {precision} {side}^3", flush=True)
        o = (side - SMALL) // 2
        mu = np.random.default_rng(side).uniform(0.95, 1.05, (side,) * 3)
        mu[o:o + SMALL, o:o + SMALL, o:o + SMALL] = core
        m = {k: v if k == "mu" else float(v.flat[0]) for k, v in media.homogeneous((1, 1, 1)).items()}
        m["mu"] = 5.1e9 * mu
        s = Solver(side, side, side, 5.0, 4e-4, precision=precision, npml=0)
        s.set_source(s.cell(o + 32, o + 32, o + 32), ricker(60.0, 4e-4, NT) + 1.0, ("txx", "tyy", "tzz", "p"))
        s.set_medium_device(m)
        z, y, x = np.meshgrid(*[np.arange(o + 26, o + 39)] * 3, indexing="ij")
        s.set_receivers((x + side * (y + side * z)).ravel(), ("vx", "qz", "txy", "p"), NT)
        s.reset()
        s.run(NT)
        t = s.traces()
        s.close()
        ref = t if ref is None else ref
        assert np.isfinite(t).all() and all(np.any(c) for c in t)
        assert np.array_equal(t, ref), side
