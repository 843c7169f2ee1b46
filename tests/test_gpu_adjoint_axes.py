"""The adjoint step on grids of one, two and three axes: the dot-product test of test_gpu_adjoint on each,
and the same cotangents on every plane of a 2D grid (the crystals turned with it)."""
import numpy as np
import pytest
import torch

import test_gpu_adjoint as T
from openphase_amd.adjoint import DeviceStates
from openphase_amd.engine import Engine, StepConfig
from openphase_amd.microstructure import Lists, voronoi_grains

pytestmark = pytest.mark.gpu


def _case(dims, precision=0):
    case = T._Case()
    kw = {k: getattr(case.cfg, k) for k in ("nphases", "sigma", "mu", "energy_model", "epsilon", "dg_mode", "dg_value")}
    case.cfg = StepConfig(*dims, precision=precision, **kw)
    case.dt = 0.9 * case.cfg.max_time_step()
    case.init = voronoi_grains(*dims, 8, seed=0x0FE4)
    return case


@pytest.mark.parametrize("dims", [(64, 0, 64), (0, 64, 64), (400, 0, 0), (0, 400, 0), (0, 0, 400), (24, 22, 26)])
def test_dot_product(dims, monkeypatch):
    print(f"adjoint step on {dims}", flush=True)
    monkeypatch.setattr(T, "_Case", lambda case=_case(dims): case)
    T.test_adjoint_step_dot_product()


def _cotangents(dims, axes, precision):
    case = _case(dims, precision)
    xy = voronoi_grains(40, 36, 0, 8, seed=0x0FE4)
    case.init = Lists(case.cfg.shape, xy.count, xy.index, xy.value)
    # the rows of a rotation are the grid's axes: row of x, of y, of z in this plane
    case.rotation = np.ascontiguousarray(np.asarray(case.rotation).reshape(-1, 3, 3)[:, axes])
    eng = case.setup(Engine(case.cfg))
    eng.step(case.dt, 5)
    st = DeviceStates(eng)
    before = st.save()
    eng.step(case.dt, 1)
    after = st.save()
    st.restore(before)
    g = torch.Generator(device="cuda").manual_seed(5)
    lam = torch.randn(st.slots, st.ncells, dtype=torch.float64, device="cuda", generator=g)
    prev = torch.empty_like(lam)
    grad = torch.zeros(12, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    eng.adjoint_step(case.dt, lam.data_ptr(), prev.data_ptr(), grad.data_ptr(), *st.list_pointers(after))
    out = st.views(before)[2].cpu().numpy(), prev.cpu().numpy(), grad.cpu().numpy()
    eng.close()
    return out


@pytest.mark.parametrize("precision", [0, 1])
def test_every_plane_gives_the_same_cotangents(precision):
    print(f"adjoint step in every plane, precision {precision}", flush=True)
    ref = _cotangents((40, 36, 0), [0, 1, 2], precision)
    # (a phase has no driving force against itself)
    assert np.abs(ref[1]).max() > 0 and np.count_nonzero(ref[2]) == 10
    # the sums along the axes differ in where a zero is added only
    for dims, axes in (((40, 0, 36), [0, 2, 1]), ((0, 40, 36), [2, 0, 1])):
        for a, b in zip(ref, _cotangents(dims, axes, precision)):
            assert np.array_equal(a, b), dims
