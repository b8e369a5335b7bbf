"""GPU checks of the adjoint's two passes where their branches meet.

* FP64 gradients against the FP64 host adjoint (scatter form, pinned on the CPU) on grids whose
  absorbing slabs fill the axis, meet in the middle, or are absent, at both orders: the derivative
  adjoints then come from the slab records, the full arrays, or both within one stencil.  The two
  differ only in summation order; the bar is the 1e-8 of the existing comparison.
* Adjoint sources: several receivers in one cell add up (a list with duplicates gives the gradient
  of the merged list: FP64, linear in the sources, 1e-10), receivers on every recorded field, on the
  first and last updated cells and on the outer planes.
"""
import numpy as np
import pytest

from biot_amd import FIELDS, Solver, _lib, configs, media, ricker
from biot_amd._lib import PARAM_NAMES
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _profiles(s):
    """The handle's own profiles as its double path holds them (e, a = -dt d / 2 at integer, then
    half nodes, through the x0.01 float storage): recomputed ones differ in the last float bit, which
    a grid that is all absorbing slab shows."""
    out, c = [], np.float32(0.01)
    for axis in range(3):
        d, d2, e, e2 = [(v * c).astype(np.float32).astype(np.float64) for v in s.pml_profile(axis)]
        dt = float(np.float32(configs.DT))
        out.append([e * 100.0, -dt * d * 100.0 * 0.5, e2 * 100.0, -dt * d2 * 100.0 * 0.5])
    return out


@pytest.mark.parametrize("order,size,npml", [(4, (20, 20, 20), 9), (2, (12, 25, 14), 5), (4, (13, 9, 70), 0),
                                             (2, (66, 11, 8), 3)])
def test_fp64_gradients_equal_host_adjoint(order, size, npml):
    import oracle

    nx, ny, nz = size
    shape, nt = (nz, ny, nx), 40
    print(f"adjoint passes order {order} {nx}x{ny}x{nz} npml {npml}", flush=True)
    rng = np.random.default_rng(4)
    p = media.params_from_medium(media.homogeneous(shape))
    p = {k: v * rng.uniform(0.95, 1.05, shape) for k, v in p.items()}
    w = ricker(60.0, configs.DT, nt) + 1.0
    src = nx // 2 + (ny // 2) * nx + (nz // 2) * nx * ny
    rec = np.sort(rng.choice(nx * ny * nz, 25, replace=False)).astype(np.int64)
    fields = ("vx", "vz", "tyz", "p")
    s = Solver(nx, ny, nz, configs.DX, configs.DT, order=order, precision="fp64", npml=npml)
    s.set_params(p)
    s.set_source(src, w, configs.SRC_EXPLOSIVE)
    s.set_receivers(rec, fields, nt)
    y = rng.standard_normal((4, nt, len(rec))).astype(np.float32)
    K = _lib.params_coefficients(nx, ny, nz, configs.DX, configs.DT, p)
    prof = _profiles(s)
    mask = sum(1 << FIELDS.index(f) for f in configs.SRC_EXPLOSIVE)
    ha = oracle.HostAdjoint(nx, ny, nz, order, prof, K, src, mask, w, rec, [FIELDS.index(f) for f in fields])
    ref, _ = ha.adjoint(nt, y.astype(np.float64), every=10)
    for every in (15, 1):
        s.forward_checkpointed(nt, every)
        _, gk = s.adjoint(y, coefs=True)
        for k, (a, b) in enumerate(zip(gk, ref)):
            e = rel_l2(np.ravel(a), np.ravel(b))
            assert e <= 1e-8, (every, _lib.KCOEF_NAMES[k], e)
    s.close()


def test_receivers_that_share_a_cell_add_up():
    nx, ny, nz, nt = 23, 18, 21, 30
    print("adjoint sources sharing cells", flush=True)
    rng = np.random.default_rng(6)
    p = media.params_from_medium(media.homogeneous((nz, ny, nx)))
    s = Solver(nx, ny, nz, 5.0, 4e-4, order=4, precision="fp64", npml=4)
    cell = s.cell
    cells = [cell(2, 2, 2), cell(nx - 3, ny - 3, nz - 3), cell(11, 9, 10), cell(11, 9, 11), cell(0, 3, 4),
             cell(nx - 1, ny - 1, nz - 1), cell(5, 1, 6)]
    fields = ("vx", "vy", "qz", "txx", "txy", "tyz", "p")
    dup = [cells[q] for q in (2, 0, 3, 2, 1, 4, 2, 5, 6, 0)]
    y = rng.standard_normal((len(fields), nt, len(dup))).astype(np.float32)
    y = np.round(y * 64) / 64  # sums of a few are exact in float32
    merged = np.zeros((len(fields), nt, len(cells)), np.float32)
    for e, c in enumerate(dup):
        merged[:, :, cells.index(c)] += y[:, :, e]
    s.set_params(p)
    s.set_source(cell(11, 9, 8), ricker(60.0, 4e-4, nt) + 1.0, ("txx", "tyy", "tzz", "p"))
    out = []
    for rec, src in ((dup, y), (cells, merged)):
        s.set_receivers(rec, fields, nt)
        s.forward_checkpointed(nt, 10)
        out.append(s.adjoint(src)[0])
    for k in PARAM_NAMES:
        assert np.any(out[0][k]) and rel_l2(out[0][k], out[1][k]) <= 1e-10, k
    s.close()
