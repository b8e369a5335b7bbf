"""GPU check of the coefficient records of media with few distinct cells.  A record holds the values
that its cells' arrays hold, and the arithmetic is the same, so a run is equal bit for bit to the run
that streams the arrays: here the run of a model whose far end has too many different cells, compared
before the wave that left the near end can have been there and back (at most 4 cells a step)."""
import numpy as np
import pytest

from biot_amd import Solver, media, ricker

pytestmark = pytest.mark.gpu

NX, NY, NZ, NT, FAR = 41, 37, 100, 18, 60


def near(kind):
    """mu of the near end: one rock, two layers, a different value in every plane, a mix of two
    rocks cell by cell.  A block of the largest value is in each, so every coefficient has its largest
    value, and with it its storage scale, from the near end."""
    mu = np.full((NZ, NY, NX), 5e9)
    if kind == "layers":
        mu[20:] = 6e9
    if kind == "planes":
        mu *= (1 + 0.001 * np.arange(NZ))[:, None, None]
    if kind == "mix":
        mu[np.random.default_rng(5).random(mu.shape) < 0.5] = 5.5e9
    mu[2, 2, 2], mu[3:6, 3:6, 3:6] = 3e9, 8e9
    return mu


@pytest.mark.parametrize("precision", ["fp32", "fp64", "fp16", "fp16t", "fp16c"])
@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("kind", ["one", "layers", "planes", "mix"])
def test_records_give_the_streamed_coefficients_run(precision, order, kind, tmp_path, monkeypatch):
    print(f"records {precision} order {order} {kind}", flush=True)
    few = media.homogeneous((NZ, NY, NX))
    few["mu"] = near(kind)
    many = dict(few)
    many["mu"] = few["mu"].copy()
    many["mu"][FAR:] *= 1 + 0.01 * np.random.default_rng(6).random((NZ - FAR, NY, NX))
    s = Solver(NX, NY, NZ, 5.0, 4e-4, order=order, precision=precision, npml=6)
    s.set_source(s.cell(20, 18, 12), ricker(60.0, 4e-4, NT) + 1.0, ("txx", "tyy", "tzz", "p"))
    s.set_receivers(np.arange(2 * NX * NY, 15 * NX * NY, 7), ("vx", "vz", "txy", "p"), NT)
    monkeypatch.setenv("BIOT_TUNE_CACHE", str(tmp_path / "tune.txt"))
    runs = []
    for medium in (few, many, few):
        s.set_medium_device(medium)
        s.reset()
        s.run(NT)
        runs.append(s.traces())
    s.autotune(1)
    s.close()
    assert np.isfinite(runs[0]).all() and all(np.any(c) for c in runs[0])
    for r in runs[1:]:
        assert np.array_equal(runs[0], r)
    # the few-cell medium did go by records: its tile shape is filed under that route
    key = (tmp_path / "tune.txt").read_text().split()
    assert key[2].endswith("r")
