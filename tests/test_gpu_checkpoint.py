"""Device checkpoints: save, step, restore gives the saved state back bit for bit, in aligned device
memory (copied by kernels) and at an odd address (copied by the runtime)."""
import numpy as np
import pytest

from openphase_amd.engine import Engine, StepConfig
from openphase_amd.microstructure import Lists
from test_gpu_deferred import _random_lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 16, 1])
@pytest.mark.parametrize("dims,pool,precision", [((1, 0, 0), 1, 0), ((9, 7, 0), 7, 1), ((7, 6, 5), 9, 0), ((3, 3, 0), 300, 0)])
def test_save_and_restore(dims, pool, precision, offset):
    import torch

    cfg = StepConfig(*dims, precision=precision, slots=12)
    lists = _random_lists(cfg.shape, pool, min(pool, 6), seed=pool)
    print(f"checkpoint {dims} pool {pool} precision {precision} offset {offset}", flush=True)
    e = Engine(cfg)
    e.set_grains(np.zeros(pool, np.int32))
    e.upload(lists)
    e.finalize_initialization()
    blob = torch.zeros(e.state_bytes() + 32, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    before, grains, records = e.download(), e.grains(), e.grain_records()
    e.save_state(blob.data_ptr() + offset)
    if np.prod(cfg.shape) > 9:
        e.step(0.3 * cfg.max_time_step(), 3)
    e.restore_state(blob.data_ptr() + offset)
    after = e.download()
    assert np.array_equal(before.count, after.count) and np.array_equal(before.index, after.index)
    assert np.array_equal(before.value, after.value)
    for a, b in zip(grains + records, e.grains() + e.grain_records()):
        assert np.array_equal(a, b)
    e.close()


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dims,pool,precision", [((1, 0, 0), 2, 0), ((9, 7, 0), 7, 1), ((3, 3, 0), 300, 0), ((3, 3, 0), 300, 1)])
def test_restore_over_another_state(dims, pool, precision, offset):
    """The context holds other lists and other grain records between save and restore (also where there
    are more grains than cells), and a blob saved from those is another blob."""
    import torch

    cfg = StepConfig(*dims, precision=precision, slots=12)
    first = _random_lists(cfg.shape, pool, min(pool, 6), seed=pool)
    # the same lists of other grains
    second = Lists(first.shape, first.count, ((first.index + pool // 2) % pool).astype(np.int32), first.value)
    print(f"restore over another state {dims} pool {pool} precision {precision} offset {offset}", flush=True)
    e = Engine(cfg)
    e.set_grains(np.zeros(pool, np.int32))

    def state():
        lists = e.download()
        return [lists.count, lists.index, lists.value, *e.grains(), *e.grain_records()]

    states, blobs = [], []
    for lists in (first, second):
        e.upload(lists)
        e.finalize_initialization()
        states.append(state())
        blobs.append(torch.zeros(e.state_bytes() + 32, dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
        e.save_state(blobs[-1].data_ptr() + offset)
    # lists, and volumes of grains beyond the number of cells among them
    ncells = int(np.prod(cfg.shape))
    assert not np.array_equal(states[0][1], states[1][1]) and not np.array_equal(states[0][3], states[1][3])
    assert pool < 300 or not np.array_equal(states[0][3][ncells:], states[1][3][ncells:])
    for i in (0, 1, 0):
        e.restore_state(blobs[i].data_ptr() + offset)
        for a, b in zip(states[i], state()):
            assert np.array_equal(a, b)
    e.close()
