"""GPU check of the tile mappings: a run does not depend on the tile shape.  Every cell is updated
by one thread with the same operations whatever the shape, so all fields are equal bit for bit,
between rectangles (by > 1), runs of consecutive cells of the plane (by = 1, rows narrower than,
equal to and wider than a run) and the shape a new handle chooses."""
import numpy as np
import pytest

from biot_amd import FIELDS, Solver, media, ricker

pytestmark = pytest.mark.gpu

SHAPES = [(64, 2, 16), (64, 1, 1), (64, 1, 5), (128, 1, 2), (256, 1, 3), (256, 1, 64)]


@pytest.mark.parametrize("precision,order,size", [("fp32", 4, (5, 5, 5)), ("fp32", 2, (3, 70, 6)),
                                                  ("fp64", 4, (63, 9, 14)), ("fp16m", 4, (64, 12, 9)),
                                                  ("fp16t", 2, (65, 31, 8)), ("fp16c", 4, (257, 7, 10)),
                                                  ("fp16", 4, (301, 11, 12))])
def test_fields_do_not_depend_on_the_tile_shape(precision, order, size):
    nx, ny, nz = size
    print(f"tile shapes {precision} order {order} {nx}x{ny}x{nz}", flush=True)
    s = Solver(nx, ny, nz, 5.0, 4e-4, order=order, precision=precision,
               npml=min(3, (min(size) - 2) // 2))
    src = s.cell(nx // 2, ny // 2, nz // 2)
    s.set_source(src, ricker(60.0, 4e-4, 25) + 1.0, ("txx", "tyy", "tzz", "p"))
    s.set_medium(media.homogeneous((nz, ny, nx)))
    s.set_receivers(np.arange(0, nx * ny * nz, 17), ("vx", "vz", "p"), 25)
    ref = None
    for shape in [None] + SHAPES:
        if shape:
            s.set_launch_shape(*shape)
        s.reset()
        s.run(25)
        got = [s.traces()] + [s.field(f, f64=True) for f in FIELDS]
        if ref is None:
            ref = got
            assert all(np.any(g) for g in got[1:4]) and np.isfinite(got[0]).all()
        for a, b in zip(ref, got):
            assert np.array_equal(a, b), shape
    s.close()
