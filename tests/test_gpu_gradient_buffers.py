"""GPU check of what gradients share from one call to the next and of how they reach the host.  A
batch whose buffers served other gradients (other data, steps, checkpoints, another model, a run on a
shot's own handle, a release in between) gives what a new batch gives: the same launches on the same
values, so the gradients are equal bit for bit (J to 1e-12: its sum's order is free).  Gradients of
sizes around the parts in which they are read back (2^18 doubles) equal the host's chain rule of the
coefficient gradients of the same call, to 1e-12 as sums of up to 30 doubles in another order do.  The
last segment's states are the forward run's own or recomputed ones, equal bit for bit: a second sweep
over the same checkpoints, which finds the first segment's states in their place, gives the same
gradients, and the run that kept them the plain run's traces and fields."""
import numpy as np
import pytest

from biot_amd import FIELDS, Solver, _lib, media, ricker
from biot_amd._lib import PARAM_NAMES
from biot_amd.batch import Batch
from conftest import rel_l2

pytestmark = pytest.mark.gpu

SHOTS = [((0, 2, 1), (24, 20, 22)), ((5, 0, 3), (19, 30, 21)), ((9, 9, 8), (27, 24, 33))]
MODEL = (40, 36, 44)


def params(seed):
    shape = MODEL[::-1]
    rng = np.random.default_rng(seed)
    p = media.params_from_medium(media.homogeneous(shape))
    return {k: v * rng.uniform(0.95, 1.05, shape) for k, v in p.items()}


def new_batch(p, precision):
    b = Batch(*MODEL, 5.0, 4e-4, precision=precision, npml=4)
    for (x, y, z), (nx, ny, nz) in SHOTS:
        win = {k: np.ascontiguousarray(v[z:z + nz, y:y + ny, x:x + nx]) for k, v in p.items()}
        rec = np.stack([np.arange(4, nx - 4), np.full(nx - 8, ny // 2), np.full(nx - 8, 5)], axis=1)
        b.add_shot((x, y, z), (nx, ny, nz), win, (nx // 2, ny // 2, nz // 2), ricker(60.0, 4e-4, 14) + 1.0, rec,
                   ("vx", "p"), ("txx", "tyy", "tzz", "p"))
    return b


def data(seed):
    rng = np.random.default_rng(seed)
    return [(0.1 * rng.standard_normal((2, 14, s[0] - 8))).astype(np.float32) for _, s in SHOTS]


@pytest.mark.parametrize("precision", ["fp32", "fp64", "fp16t", "fp16m"])
def test_batch_buffers_serve_the_next_gradient(precision):
    print(f"batch gradient buffers {precision}", flush=True)
    b = new_batch(params(1), precision)
    steps = [(1, 14, 5, 7), (1, 14, 5, 8), (1, 14, 4, 8), (1, 11, 4, 8), (2, 11, 4, 8), (2, 14, 20, 9), (1, 14, 5, 7)]
    model = 1
    for i, (m, nt, every, obs) in enumerate(steps):
        if m != model:
            b.set_model(params(m))
            model = m
        if i == 5:
            b.release()
        b.forward(nt, graph_steps=0)
        plain = [b.traces(k) for k in range(len(SHOTS))]
        J, g = b.gradient(nt, data(obs), every=every)
        for k, t in enumerate(plain):
            assert np.any(t) and np.array_equal(b.traces(k), t), (i, k)
        fresh = new_batch(params(m), precision)
        J0, g0 = fresh.gradient(nt, data(obs), every=every)
        fresh.close()
        assert abs(J - J0) <= 1e-12 * J0, i
        for k in PARAM_NAMES:
            assert np.any(g0[k]) and np.array_equal(g[k], g0[k]), (i, k)
    b.close()


@pytest.mark.parametrize("size", [(64, 64, 64), (65, 64, 67), (33, 20, 19), (90, 81, 72)])
def test_gradients_read_back_whole(size):
    nx, ny, nz = size
    nt = 14
    print(f"gradients read back {nx}x{ny}x{nz}", flush=True)
    rng = np.random.default_rng(8)
    p = {k: v * rng.uniform(0.9, 1.1, (nz, ny, nx))
         for k, v in media.params_from_medium(media.homogeneous((nz, ny, nx))).items()}
    s = Solver(nx, ny, nz, 5.0, 4e-4, precision="fp32", npml=4)
    s.set_source(s.cell(nx // 2, ny // 2, nz - 5), ricker(60.0, 4e-4, nt) + 1.0, ("txx", "tyy", "tzz", "p"))
    s.set_params(p)
    s.set_receivers(rng.choice(nx * ny * nz, 400, replace=False), ("vx", "vz", "p"), nt)
    s.forward_checkpointed(nt, 7)
    y = rng.standard_normal((3, nt, 400)).astype(np.float32)
    g, gk = s.adjoint(y, params=True, coefs=True)
    s.close()
    ref = _lib.params_chain(nx, ny, nz, 5.0, 4e-4, p, gk)
    for k, r in zip(PARAM_NAMES, ref):
        assert np.any(r.ravel()[-nx * ny * 4:]) and rel_l2(g[k].ravel(), r) <= 1e-12, k


@pytest.mark.parametrize("precision,every", [("fp32", 7), ("fp64", 5), ("fp16t", 14), ("fp16m", 20), ("fp16", 13),
                                             ("fp16c", 6)])
def test_last_segment_of_the_forward_run_serves_the_sweep(precision, every):
    nx, ny, nz, nt = 34, 25, 29, 14
    print(f"last segment {precision} every {every}", flush=True)
    rng = np.random.default_rng(3)
    p = {k: v * rng.uniform(0.9, 1.1, (nz, ny, nx))
         for k, v in media.params_from_medium(media.homogeneous((nz, ny, nx))).items()}
    s = Solver(nx, ny, nz, 5.0, 4e-4, precision=precision, npml=4)
    s.set_source(s.cell(nx // 2, ny // 2, nz // 2), ricker(60.0, 4e-4, nt) + 1.0, ("txx", "tyy", "tzz", "p"))
    s.set_params(p)
    s.set_receivers(rng.choice(nx * ny * nz, 40, replace=False), ("vx", "vz", "p"), nt)
    s.reset()
    s.run(nt)
    plain = [s.traces()] + [s.field(f, f64=True) for f in FIELDS]
    y = rng.standard_normal((3, nt, 40)).astype(np.float32)
    first = None
    for _ in range(2):  # the second run in the buffers of the first
        s.forward_checkpointed(nt, every)
        for a, b in zip(plain, [s.traces()] + [s.field(f, f64=True) for f in FIELDS]):
            assert np.array_equal(a, b)
        for _ in range(2):
            g = s.adjoint(y)[0]
            first = first or g
            for k in PARAM_NAMES:
                assert np.any(g[k]) and np.array_equal(g[k], first[k]), k
    s.close()
