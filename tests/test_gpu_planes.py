"""2D grids in every plane, isotropic and with orientation-dependent energies and a driving force: the step
kernel's tiles (those staged whole and those that march along x, with remainders on both axes) against
the per-cell kernel bit for bit, and that one against the oracle."""
import numpy as np
import pytest

from openphase_amd.engine import Engine
from openphase_amd.microstructure import random_rotations, voronoi_grains
import oracle as O
from test_gpu_deferred import _config

pytestmark = pytest.mark.gpu

STEPS, GRAINS = 6, 14


def _run(make, cfg, lists, tile=None):
    _, rot = random_rotations(GRAINS, seed=9)
    e = make(cfg)
    if tile:
        e.set_tile_shape(*tile)
    e.set_grains(np.arange(GRAINS, dtype=np.int32) % cfg.nphases, rot)
    e.upload(lists)
    e.finalize_initialization()
    e.step(0.9 * cfg.max_time_step(), STEPS)
    out = e.download(), e.grains()[0]
    e.close()
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("model", ["iso", "cubic"])
@pytest.mark.parametrize("dims", [(83, 70, 0), (83, 0, 70), (0, 83, 70)])
def test_tiles_of_every_plane(dims, model, precision):
    cfg = _config(model, dims, precision)
    lists = voronoi_grains(*dims, GRAINS, seed=77)
    if dims[0] == 0:
        tiles = [(0, 0, 0), (1, 16, 16), (1, 8, 32), (1, 4, 64)]
    else:
        tiles = [(0, 0, 0)] + [(rows, *((width, 1) if dims[1] else (1, width))) for width in (16, 32, 64) for rows in (1, 4, 8, 16)]
    ref, volume = _run(Engine, cfg, lists, (-1,))
    for tile in tiles:
        print(f"{model} {dims} precision {precision} tile {tile}", flush=True)
        got, vol = _run(Engine, cfg, lists, tile)
        assert np.array_equal(got.count, ref.count) and np.array_equal(got.index, ref.index), tile
        assert np.array_equal(got.value, ref.value) and np.array_equal(vol, volume), tile
    if precision == 0:
        exp, _ = _run(O.Oracle, cfg, lists)
        assert np.array_equal(ref.count, exp.count) and np.array_equal(ref.index, exp.index)
        if model == "iso":
            assert np.array_equal(ref.value, exp.value)
        else:
            # the pair energy's fourth power and tanh differ in the last bit (1e-12 bounds a step's values)
            assert np.abs(ref.value - exp.value).max() <= STEPS * 1e-12
