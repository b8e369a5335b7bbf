"""GPU check of the runs of states the adjoint steps through (each step reads one state and writes the
next): traces, final fields and the gradients' states are those of the steps in place.  A stored run
(every = 1) equals a plain run bit for bit, and gives the gradients of recomputed segments bit for
bit, for sources the stress launch adds, a source a receiver samples, one on the outer planes (which
no half step writes: its value is carried along, past the wavelet's end too) and one on the first
updated cell; a second run in the same buffers gives the same again."""
import numpy as np
import pytest

from biot_amd import FIELDS, Solver, media, ricker
from biot_amd._lib import PARAM_NAMES

pytestmark = pytest.mark.gpu

NX, NY, NZ, NT = 34, 15, 19, 23
SOURCES = {"inside": (17, 7, 9), "recorded": (17, 7, 9), "outer plane": (17, 7, 1), "first": (2, 2, 2)}
CASES = [("fp32", n) for n in SOURCES] + [(p, n) for p in ("fp16", "fp16t", "fp16c", "fp16m", "fp64")
                                          for n in ("inside", "outer plane")]


@pytest.mark.parametrize("precision,name", CASES)
def test_stored_run_equals_plain_run(precision, name):
    print(f"state runs {precision}: {name}", flush=True)
    rng = np.random.default_rng(2)
    p = media.params_from_medium(media.homogeneous((NZ, NY, NX)))
    p = {k: v * rng.uniform(0.95, 1.05, v.shape) for k, v in p.items()}
    s = Solver(NX, NY, NZ, 5.0, 4e-4, order=4, precision=precision, npml=3)
    src = s.cell(*SOURCES[name])
    s.set_source(src, ricker(60.0, 4e-4, NT - 8) + 1.0, ("txx", "tyy", "tzz", "p"))
    s.set_params(p)
    rec = np.arange(3, NX * NY * NZ, 77)
    s.set_receivers(np.append(rec[rec != src], [src] if name == "recorded" else []), ("vx", "txx", "p"), NT)
    s.reset()
    s.run(NT)
    plain = [s.traces()] + [s.field(f, f64=True) for f in FIELDS]
    assert np.any(plain[1]) and np.isfinite(plain[0]).all()
    y = rng.standard_normal(plain[0].shape).astype(np.float32)
    grads = []
    for every in (1, 1, 50, 50):
        s.forward_checkpointed(NT, every)
        for a, b in zip(plain, [s.traces()] + [s.field(f, f64=True) for f in FIELDS]):
            assert np.array_equal(a, b), every
        grads.append(s.adjoint(y, coefs=True))
    # one segment of 50 steps and a stored run add their float partial sums alike
    for g in grads[1:]:
        for k in PARAM_NAMES:
            assert np.any(g[0][k]) and np.array_equal(g[0][k], grads[0][0][k]), k
    s.close()
