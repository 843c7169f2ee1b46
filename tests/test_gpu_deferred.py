"""The deferred-cell kernel on every list length it takes: random lists drawn from a small pool of
grains give merged lists of up to the pool's size (2 to 16), against the CPU oracle."""
import numpy as np
import pytest

from openphase_amd import _capi
from openphase_amd.engine import Engine, StepConfig
from openphase_amd.microstructure import Lists, random_rotations
import oracle as O

pytestmark = pytest.mark.gpu


def _random_lists(shape, pool, longest, seed):
    """Cells of 1 to `longest` entries in random order with values summing to 1; a third are bulk."""
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    count = np.where(rng.random(n) < 1 / 3, 1, rng.integers(1, longest + 1, n)).astype(np.int32)
    index = np.concatenate([rng.permutation(pool)[:c] for c in count]).astype(np.int32)
    value = np.concatenate([rng.dirichlet(np.ones(c)) for c in count])
    return Lists(shape, count, index, value)


def _config(model, dims, precision=0):
    kw = dict(slots=16 if precision == 0 else 15, precision=precision, nucleus_volume_factor=1e-3)
    if model != "iso":
        kw.update(nphases=2, sigma=np.array([[0.24, 0.3], [0.3, 0.2]]), mu=np.array([[4e-9, 3e-9], [3e-9, 4e-9]]))
    if model == "tj":
        kw.update(tj_model=_capi.MPF_TJ_VALUE, tj_energy=0.1)
    if model == "cubic":
        kw.update(energy_model=np.full((2, 2), _capi.MPF_ENERGY_CUBIC, np.int32), epsilon=np.full((2, 2), 0.05),
                  dg_mode=np.array([[0, 1], [1, 0]], np.int32), dg_value=np.array([[0.0, 1e5], [-1e5, 0.0]]))
    return StepConfig(*dims, **kw)


def _step(make, cfg, lists, pool, dt):
    _, rot = random_rotations(pool, seed=3)
    e = make(cfg)
    e.set_grains(np.arange(pool, dtype=np.int32) % cfg.nphases, rot)
    e.upload(lists)
    e.finalize_initialization()
    e.step(dt, 1)
    out = e.download(), e.limiter_warnings()
    e.close()
    return out


def _dense(lists, pool):
    out = np.zeros((lists.ncells, pool))
    out[np.repeat(np.arange(lists.ncells), lists.count), lists.index] = lists.value
    return out


@pytest.mark.parametrize("model", ["iso", "two", "tj", "cubic"])
@pytest.mark.parametrize("dims,pool,longest", [((9, 7, 0), 2, 2), ((9, 7, 0), 7, 3), ((7, 6, 5), 5, 5), ((7, 6, 5), 8, 8),
                                               ((7, 6, 5), 9, 4), ((5, 6, 7), 16, 9)])
def test_lists_of_every_length(model, dims, pool, longest):
    cfg = _config(model, dims)
    lists = _random_lists(cfg.shape, pool, longest, seed=11 * pool + longest)
    dt = 0.5 * cfg.max_time_step()
    print(f"{model} {dims} pool {pool} longest {longest}", flush=True)
    got, warn = _step(Engine, cfg, lists, pool, dt)
    exp, warn_exp = _step(O.Oracle, cfg, lists, pool, dt)
    assert np.array_equal(got.count, exp.count) and np.array_equal(got.index, exp.index)
    if model == "cubic":
        # the pair energy's fourth power and tanh differ in the last bit (1e-12 bounds a step's values)
        assert np.abs(got.value - exp.value).max() <= 1e-12
    else:
        assert np.array_equal(got.value, exp.value)
        assert warn == warn_exp


@pytest.mark.parametrize("model,precision", [("two", 0), ("cubic", 0), ("iso", 1)])
@pytest.mark.parametrize("dims,pool,longest", [((9, 7, 0), 4, 3), ((7, 6, 5), 8, 8), ((5, 6, 7), 15, 9)])
def test_energy_and_flags(model, precision, dims, pool, longest):
    """The interface energy on lists of every length, with the pairs of the current state and of the
    one before the step, and the downloaded flags."""
    cfg = _config(model, dims, precision)
    lists = _random_lists(cfg.shape, pool, longest, seed=7 * pool + longest)
    if precision:
        lists.value[:] = lists.value.astype(np.float32)
    _, rot = random_rotations(pool, seed=3)
    print(f"energy {model} precision {precision} {dims} pool {pool}", flush=True)
    eng, orc = Engine(cfg), O.Oracle(_config(model, dims))
    for e in (eng, orc):
        e.set_grains(np.arange(pool, dtype=np.int32) % cfg.nphases, rot)
        e.upload(lists)
        e.finalize_initialization()
        if e is orc:
            orc.keep_step_start(True)
        e.step(0.5 * cfg.max_time_step(), 1)
    # sums of about 10^4 terms of either sign, FP32 states with 24-bit values
    rel = 1e-11 if precision == 0 else 1e-4
    for ip in ("current", "previous"):
        assert eng.interface_energy(ip) == pytest.approx(orc.interface_energy(ip), rel=rel)
    got, flags = eng.download(with_flags=True)
    exp, flags_exp = orc.download(with_flags=True)
    if precision == 0:
        assert np.array_equal(got.count, exp.count) and np.array_equal(flags, flags_exp)
    eng.close()
    orc.close()


@pytest.mark.parametrize("pool,longest", [(3, 3), (8, 5), (15, 9)])
def test_single_precision_lists(pool, longest):
    cfg = _config("two", (7, 6, 5), precision=1)
    lists = _random_lists(cfg.shape, pool, longest, seed=5 * pool + longest)
    dt = 0.5 * cfg.max_time_step()
    print(f"fp32 pool {pool} longest {longest}", flush=True)
    got, _ = _step(Engine, cfg, lists, pool, dt)
    exp, _ = _step(O.Oracle, _config("two", (7, 6, 5)), lists, pool, dt)
    # one step in FP32: increments of order 1 with 24-bit terms that cancel to a few per cent
    assert np.abs(_dense(got, pool) - _dense(exp, pool)).max() <= 1e-5


# the entry an FP32 list holds implicitly (the largest) beyond the eighth slot
@pytest.mark.parametrize("longest", [9, 15])
def test_single_precision_lists_with_a_late_implicit_entry(longest):
    cfg = _config("two", (7, 6, 5), precision=1)
    lists = _random_lists(cfg.shape, 15, longest, seed=longest)
    off = lists.offsets()
    for c in np.flatnonzero(lists.count > 8):
        v = lists.value[off[c]:off[c + 1]]
        v.sort()
    dt = 0.5 * cfg.max_time_step()
    print(f"fp32 late implicit entry, longest {longest}", flush=True)
    got, _ = _step(Engine, cfg, lists, 15, dt)
    exp, _ = _step(O.Oracle, _config("two", (7, 6, 5)), lists, 15, dt)
    # one step in FP32: increments of order 1 with 24-bit terms that cancel to a few per cent
    assert np.abs(_dense(got, 15) - _dense(exp, 15)).max() <= 1e-5


def _vanishing(grains):
    """9 x 9 cells, an interface of grains 0 and 1 along x, and around cell (4, 4) sixteen entries of
    `grains` other grains so small that the next step erases most of them: that cell's merged list is
    `grains` + 2 long before the step and shorter after it."""
    lists, n = [], 0
    for x in range(9):
        for y in range(9):
            cell = {0: 1.0} if x <= 4 else ({0: 0.5, 1: 0.5} if x == 5 else {1: 1.0})
            if max(abs(x - 4), abs(y - 4)) == 1:
                for _ in range(2):
                    cell[2 + n % grains] = 1e-5
                    n += 1
                cell[max(cell, key=cell.get)] -= 2e-5
            lists.append(cell)
    return Lists((9, 9, 1), np.array([len(c) for c in lists], np.int32), np.array([g for c in lists for g in c], np.int32),
                 np.array([v for c in lists for v in c.values()]))


@pytest.mark.parametrize("model", ["iso", "two"])
def test_energy_of_a_vanished_list(model):
    """Energies with the pairs of the state before the step, where one list was long (16 entries of other
    grains in the box, 12 grains merged), against the oracle."""
    cfg = _config(model, (9, 9, 0))
    lists = _vanishing(10)
    eng, orc = Engine(cfg), O.Oracle(cfg)
    for e in (eng, orc):
        e.set_grains(np.arange(12, dtype=np.int32) % cfg.nphases)
        e.upload(lists)
        e.finalize_initialization()
        if e is orc:
            orc.keep_step_start(True)
        e.step(cfg.max_time_step(), 1)
    assert np.array_equal(eng.download().index, orc.download().index)
    for ip in ("previous", "current"):
        # sums of about 100 terms
        assert eng.interface_energy(ip) == pytest.approx(orc.interface_energy(ip), rel=1e-12)
    eng.close()
    orc.close()


@pytest.mark.parametrize("model", ["iso", "two", "cubic"])
def test_energy_refuses_a_list_no_step_takes(model):
    """18 grains merged in one cell: the step reports the cell, and so does the energy with the pairs of
    the state before that step, for every form of the tables; the lists after it are short enough."""
    cfg = _config(model, (9, 9, 0))
    _, rot = random_rotations(18, seed=3)
    e = Engine(cfg)
    e.set_grains(np.arange(18, dtype=np.int32) % cfg.nphases, rot)
    e.upload(_vanishing(16))
    e.finalize_initialization()
    with pytest.raises(_capi.MpfError) as err:
        e.step(cfg.max_time_step(), 1)
    assert err.value.status == _capi.MPF_SLOT_OVERFLOW and e.overflow_cell() == 4 * 9 + 4
    assert e.interface_energy("current") > 0.0
    with pytest.raises(_capi.MpfError) as err:
        e.interface_energy("previous")
    assert err.value.status == _capi.MPF_SLOT_OVERFLOW
    e.close()
