"""GPU check of the device chain rule: the parameter gradients of biot_adjoint equal the host
chain rule (biot_params_chain) of the coefficient gradients of the same call.  Both evaluate the
same terms in double, up to 30 a cell summed in different orders, so they agree to a few 1e-15 of
the largest term; the bar is 1e-12 of the gradient's norm.  The grids hold the smallest one that
order 4 takes (5 cells an axis), odd sizes, and fluid cells (mu = 0 and C1 = 0, whose zero guards
drop terms)."""
import numpy as np
import pytest

from biot_amd import Solver, _lib, media, ricker
from biot_amd._lib import PARAM_NAMES
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,order,size", [("fp32", 4, (5, 5, 5)), ("fp64", 4, (37, 19, 23)),
                                                  ("fp32", 2, (3, 33, 9)), ("fp16m", 4, (65, 8, 17))])
def test_parameter_gradients_equal_host_chain_of_coefficient_gradients(precision, order, size):
    nx, ny, nz = size
    shape, nt = (nz, ny, nx), 12
    print(f"device chain {precision} order {order} {nx}x{ny}x{nz}", flush=True)
    rng = np.random.default_rng(8)
    p = media.params_from_medium(media.homogeneous(shape))
    p = {k: v * rng.uniform(0.9, 1.1, shape) for k, v in p.items()}
    fluid = rng.random(shape) < 0.1
    p["mu"] = np.where(fluid, 0.0, p["mu"])
    p["C1"] = np.where(fluid, 0.0, p["C1"])
    s = Solver(nx, ny, nz, 5.0, 4e-4, order=order, precision=precision,
               npml=min(2, (min(size) - 2) // 2))
    s.set_source(s.cell(nx // 2, ny // 2, nz // 2), ricker(60.0, 4e-4, nt) + 1.0, ("txx", "tyy", "tzz", "p"))
    s.set_params(p)
    s.set_receivers(rng.choice(nx * ny * nz, 9, replace=False), ("vx", "vz", "p"), nt)
    for every in (5, 1):
        s.forward_checkpointed(nt, every)
        y = rng.standard_normal((3, nt, 9)).astype(np.float32)
        for _ in range(2):  # the second call finds the parameters on the device
            g, gk = s.adjoint(y, params=True, coefs=True)
            ref = _lib.params_chain(nx, ny, nz, 5.0, 4e-4, p, gk)
            for k, r in zip(PARAM_NAMES, ref):
                assert np.any(r) and rel_l2(g[k].ravel(), r) <= 1e-12, k
    s.close()
