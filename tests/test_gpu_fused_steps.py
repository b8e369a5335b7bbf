"""GPU check of the work that rides on the half-step launches: a run of many steps in one call
(sources and receivers on the half steps) equals the same steps one call each (their own launches)
bit for bit - traces and all fields - and a batch equals its shots' single grids.  The layouts are
the ones where the order matters or the ride is refused: a receiver at the source cell, sources on
velocities, a source outside the update box, a wavelet or trace length that ends inside the run, no
receivers."""
import numpy as np
import pytest

from biot_amd import FIELDS, Solver, media, ricker
from biot_amd.batch import Batch
from conftest import rel_l2

pytestmark = pytest.mark.gpu

NX, NY, NZ, NT = 37, 20, 26, 24
EXPL = ("txx", "tyy", "tzz", "p")
# (source cell, source fields, receiver at the source, recorded fields, wavelet steps, trace steps)
LAYOUTS = {
    "plain": ((18, 10, 13), EXPL, False, ("vx", "vz", "p"), NT, NT),
    "receiver at the source": ((18, 10, 13), EXPL, True, ("vx", "txx", "p"), NT, NT),
    "receiver at the source, other fields": ((18, 10, 13), ("txy",), True, ("vz", "tyz", "p"), NT, NT),
    "velocity source": ((18, 10, 13), ("vx", "qz", "p"), False, ("vx", "p"), NT, NT),
    "velocity source, recorded": ((18, 10, 13), ("vx", "p"), True, ("vx", "vz", "p"), NT, NT),
    "outside the update box": ((18, 10, 1), EXPL, False, ("vx", "vz", "p"), NT, NT),
    "first updated cell": ((2, 2, 2), EXPL, False, ("qx", "vz", "tyz"), NT, NT),
    "last updated cell": ((NX - 3, NY - 3, NZ - 3), EXPL, False, ("qx", "vz", "tyz"), NT, NT),
    "short wavelet": ((18, 10, 13), EXPL, False, ("vx", "p"), 7, NT),
    "short traces": ((18, 10, 13), EXPL, False, ("vx", "p"), NT, 9),
    "velocities only": ((18, 10, 13), EXPL, False, ("vx", "qy"), NT, NT),
    "stresses only": ((18, 10, 13), EXPL, False, ("txz", "p"), NT, NT),
    "no receivers": ((18, 10, 13), EXPL, False, (), NT, 0),
}
CASES = [("fp32", name) for name in LAYOUTS] + [(p, n) for p in ("fp16", "fp16t", "fp16c", "fp16m", "fp64")
                                                for n in ("plain", "receiver at the source")]


@pytest.mark.parametrize("precision,name", CASES)
def test_one_call_equals_one_call_a_step(precision, name):
    cell, src_fields, at_source, rec_fields, nw, nt_max = LAYOUTS[name]
    print(f"fused steps {precision}: {name}", flush=True)
    s = Solver(NX, NY, NZ, 5.0, 4e-4, order=4, precision=precision, npml=4)
    src = s.cell(*cell)
    s.set_source(src, ricker(60.0, 4e-4, nw) + 1.0, src_fields)
    s.set_medium(media.homogeneous((NZ, NY, NX)))
    if rec_fields:
        cells = np.arange(5, NX * NY * NZ, 61)
        cells = np.append(cells[cells != src], [src] if at_source else [])
        s.set_receivers(cells, rec_fields, nt_max)
    out = []
    for calls in ([1] * NT, [NT], [10, 1, NT - 11]):
        s.reset()
        for n in calls:
            s.run(n)
        assert s.step() == NT
        out.append(([s.traces()] if rec_fields else []) + [s.field(f, f64=True) for f in FIELDS])
    assert np.any(out[0][-1]) and np.isfinite(out[0][-1]).all()
    for got in out[1:]:
        for a, b in zip(out[0], got):
            assert np.array_equal(a, b)
    s.close()


@pytest.mark.parametrize("at_source", [False, True])
def test_batch_equals_single_grids_with_a_receiver_at_the_source(at_source):
    print(f"fused batch, receiver at the source: {at_source}", flush=True)
    w = ricker(60.0, 4e-4, NT) + 1.0
    sizes = [(NX, NY, NZ), (20, 33, 17)]
    b = Batch(40, 40, 40, 5.0, 4e-4, order=4, precision="fp32", npml=4)
    refs = []
    for q, (nx, ny, nz) in enumerate(sizes):
        p = media.params_from_medium(media.homogeneous((nz, ny, nx)))
        src = (nx // 2, ny // 2, nz // 2)
        rec = [(3, 4, 5), (nx - 4, ny // 2, 4), src if at_source and q else (5, 5, 5)]
        b.add_shot((q, 0, 0), (nx, ny, nz), p, src, w, rec, ("vx", "txx", "p"), EXPL)
        s = Solver(nx, ny, nz, 5.0, 4e-4, order=4, precision="fp32", npml=4)
        s.set_params(p)
        s.set_source(s.cell(*src), w, EXPL)
        s.set_receivers([s.cell(*r) for r in rec], ("vx", "txx", "p"), NT)
        for _ in range(NT):
            s.run(1)
        refs.append(s.traces())
        s.close()
    for replay in range(3):
        for graph_steps in (0, 7, 8):  # 8: the run ends with a graph
            b.forward(NT, graph_steps=graph_steps)
            assert max(rel_l2(b.traces(q), r) for q, r in enumerate(refs)) <= 1e-7
    b.forward(10, graph_steps=4)  # shorter than the wavelet: no source after the last step
    short = b.traces(0)[:, :10].copy()
    assert rel_l2(short, refs[0][:, :10]) <= 1e-7 and not np.any(b.traces(0)[:, 10:])
    b.close()
