"""Averaging over the interface (driving force, curvature) with a wavefront per cell (small grids, large
spheres) and on staged tiles: ragged grids, every reach, lists of up to six entries, against the oracle."""
import numpy as np
import pytest

from openphase_amd.engine import Engine, StepConfig
import oracle as O
from test_gpu_deferred import _random_lists, _step
from test_gpu_deferred import _dense

pytestmark = pytest.mark.gpu

# a step's values: the limiter's tanh differs in the last bit between device and host
TOL = 1e-12


def _compare(cfg, pool, longest, seed):
    lists = _random_lists(cfg.shape, pool, longest, seed)
    dt = 0.3 * cfg.max_time_step()
    got, _ = _step(Engine, cfg, lists, pool, dt)
    exp, _ = _step(O.Oracle, cfg, lists, pool, dt)
    assert np.array_equal(got.count, exp.count) and np.array_equal(got.index, exp.index)
    assert np.abs(got.value - exp.value).max() <= TOL


# spheres of one chunk of offsets, of several, and longer than the grid
@pytest.mark.parametrize("dims,reach", [((33, 19, 0), 3), ((12, 50, 0), 5), ((9, 8, 10), 3), ((13, 9, 10), 5), ((12, 9, 11), 6),
                                        ((9, 10, 11), 9), ((40, 0, 0), 4)])
@pytest.mark.parametrize("weights", [0, 1, 2])
def test_driving_force(dims, reach, weights):
    cfg = StepConfig(*dims, nphases=2, sigma=np.full((2, 2), 0.24), mu=np.full((2, 2), 4e-9), slots=16,
                     nucleus_volume_factor=1e-3, dg_mode=np.array([[0, 1], [1, 0]], np.int32),
                     dg_value=np.array([[0.0, 1e5], [-7e4, 0.0]]), dg_average=True, dg_range=reach, dg_threshold=0.05,
                     dg_weights=weights)
    print(f"driving force {dims} range {reach} weights {weights}", flush=True)
    _compare(cfg, 7, 6, seed=17 * reach + weights)


@pytest.mark.parametrize("dims,reach", [((33, 19, 0), 2), ((12, 50, 0), 6), ((9, 8, 10), 3), ((13, 9, 10), 4), ((9, 10, 11), 9)])
def test_curvature(dims, reach):
    cfg = StepConfig(*dims, slots=16, nucleus_volume_factor=1e-3, regularization=True, regularization_factor=1.5,
                     curvature_factor=0.7, reg_range=reach, reg_threshold=0.02)
    print(f"curvature {dims} range {reach}", flush=True)
    _compare(cfg, 7, 6, seed=23 * reach)


@pytest.mark.parametrize("dims,reach", [((521, 509, 0), 3), ((67, 61, 65), 2)])
def test_curvature_on_tiles(dims, reach):
    # at least 2^18 cells: the averages are formed on staged tiles, here with remainders on every axis
    cfg = StepConfig(*dims, slots=16, nucleus_volume_factor=1e-3, regularization=True, regularization_factor=1.5,
                     curvature_factor=0.7, reg_range=reach, reg_threshold=0.02)
    print(f"curvature on tiles {dims} range {reach}", flush=True)
    _compare(cfg, 4, 3, seed=23 * reach)


@pytest.mark.parametrize("weights", [0, 1, 2])
def test_driving_force_on_tiles(weights):
    cfg = StepConfig(521, 509, 0, nphases=2, sigma=np.full((2, 2), 0.24), mu=np.full((2, 2), 4e-9), slots=16,
                     nucleus_volume_factor=1e-3, dg_mode=np.array([[0, 1], [1, 0]], np.int32),
                     dg_value=np.array([[0.0, 1e5], [-7e4, 0.0]]), dg_average=True, dg_range=3, dg_threshold=0.05,
                     dg_weights=weights)
    print(f"driving force on tiles, weights {weights}", flush=True)
    _compare(cfg, 4, 3, seed=31)


# grids of at least 2^18 cells with remainders on every axis, of one, two and three axes, and lists of up to
# six entries (beyond the four grains a staged cell holds)
TILED = [((521, 509, 0), 4), ((521, 0, 509), 3), ((0, 521, 509), 2), ((262149, 0, 0), 128), ((67, 61, 65), 3), ((67, 61, 65), 4)]


def _driving(dims, reach, weights, precision=0):
    return StepConfig(*dims, nphases=2, sigma=np.full((2, 2), 0.24), mu=np.full((2, 2), 4e-9), slots=8,
                      nucleus_volume_factor=1e-3, dg_mode=np.array([[0, 1], [1, 0]], np.int32),
                      dg_value=np.array([[0.0, 1e5], [-7e4, 0.0]]), dg_average=True, dg_range=reach, dg_threshold=0.05,
                      dg_weights=weights, precision=precision)


@pytest.mark.parametrize("dims,reach", TILED)
def test_driving_force_of_long_lists_on_tiles(dims, reach):
    print(f"driving force of long lists on tiles {dims} range {reach}", flush=True)
    _compare(_driving(dims, reach, reach % 3), 7, 6, seed=41 * reach)


@pytest.mark.parametrize("dims,reach", TILED)
def test_curvature_of_long_lists_on_tiles(dims, reach):
    cfg = StepConfig(*dims, slots=8, nucleus_volume_factor=1e-3, regularization=True, regularization_factor=1.5,
                     curvature_factor=0.7, reg_range=reach, reg_threshold=0.02)
    print(f"curvature of long lists on tiles {dims} range {reach}", flush=True)
    _compare(cfg, 7, 6, seed=43 * reach)


@pytest.mark.parametrize("dims,reach", [TILED[0], TILED[4], ((33, 19, 0), 3)])
def test_single_precision_driving_force(dims, reach):
    """FP32 lists, on tiles and with a wavefront per cell. The values are multiples of 2^-16 that sum to 1,
    which both precisions hold exactly: the weights are the same and the same terms count."""
    lists = _random_lists((dims[0] or 1, dims[1] or 1, dims[2] or 1), 7, 6, seed=47 * reach)
    first = np.cumsum(lists.count) - lists.count
    v = np.maximum(np.floor(lists.value * 65536), 1.0)
    v[first] += 65536 - np.add.reduceat(v, first)
    lists.value[:] = v / 65536
    assert lists.value.min() > 0
    print(f"fp32 driving force {dims} range {reach}", flush=True)
    dt = 0.3 * _driving(dims, reach, 0).max_time_step()
    got, _ = _step(Engine, _driving(dims, reach, 0, precision=1), lists, 7, dt)
    exp, _ = _step(O.Oracle, _driving(dims, reach, 0), lists, 7, dt)
    # one step in FP32: increments of order 1 with 24-bit terms that cancel to a few per cent
    assert np.abs(_dense(got, 7) - _dense(exp, 7)).max() <= 1e-5
