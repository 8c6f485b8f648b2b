"""The transport rounds' builds and their wave-level bookkeeping change no bit: the build
for one material (tables in LDS) against the general one, and the stack in which a wave's
Moller interactions wait, empty, in use and full."""

from __future__ import annotations

from dataclasses import dataclass

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@dataclass
class TwoEqualRows:
    """A one-material source's tables with the row twice: the same physics, but two rows,
    so the rounds take their general build."""

    inner: object

    @property
    def n_materials(self):
        return 2

    @property
    def provenance(self):
        return self.inner.provenance

    def build_tables(self, **kw):
        t = self.inner.build_tables(**kw)
        for name, value in list(vars(t).items()):
            a = np.asarray(value)
            if name != "majorant" and a.ndim == 2 and a.shape[0] == 1:
                object.__setattr__(t, name, np.concatenate([a, a]))
        return t


def _same(a, b):
    np.testing.assert_array_equal(a.dose, b.dose)
    np.testing.assert_array_equal(a.dose_sigma, b.dose_sigma)
    assert (a.energy_deposited, a.energy_escaped, a.energy_unscored) == (
        b.energy_deposited, b.energy_escaped, b.energy_unscored)
    assert a.counters["electron_steps"] == b.counters["electron_steps"]


# Odd extents, a run shorter than a wave's first block, deposits spread (the rounds'
# general scoring), Gaussian scattering and the kerma mode.
@pytest.mark.parametrize("shape, histories, options", [
    ((17, 9, 33), 40, {}),
    ((17, 9, 33), 60_000, {}),
    ((16, 16, 16), 60_000, dict(deposit_resolution_cm=0.07)),
    ((5, 31, 20), 60_000, dict(msc_model="gaussian")),
    ((16, 16, 16), 60_000, dict(transport_electrons=False)),
])
def test_one_material_build_equals_the_general_one(shape, histories, options):
    from pyradmc_amd import AnalyticCrossSections, HipEngine, PencilBeamSource, VoxelGrid

    density = np.random.default_rng(3).uniform(0.2, 1.9, shape)
    grid = VoxelGrid(shape=shape, spacing=(0.4, 0.5, 0.3), density=density, material=np.zeros(shape, dtype=np.int32))
    xs = AnalyticCrossSections(geometry_densities=grid.max_density_by_material())
    source = PencilBeamSource(6.0, (shape[0] * 0.2, shape[1] * 0.25, -1.0), (0.0, 0.0, 1.0))
    one = HipEngine(grid, xs).run(source, histories, 4, seed=9, **options)
    two = HipEngine(grid, TwoEqualRows(xs)).run(source, histories, 4, seed=9, **options)
    _same(one, two)
    assert one.energy_deposited > 0.0


# Electrons far above a low cutoff meet a Moller interaction in many lanes of a pass and
# leave about thirty delta electrons each, in up to seven generations; photons of 18 MeV
# bring positrons.
@pytest.mark.parametrize("rows", (1, 2))
@pytest.mark.parametrize("kind, energy, ecut, histories", [("electron", 6.0, 0.01, 4096),
                                                           ("photon", 18.0, 0.02, 40_000)])
def test_wave_stacks_of_any_size_equal_none(rows, kind, energy, ecut, histories):
    """Both builds' electron rounds against themselves without stacks (every Moller
    interaction in place, every delta electron through the queue), with the stacks whole,
    with so few slots that lanes find them full at every batch, and with one of the two."""
    from pyradmc_amd import AnalyticCrossSections, HipEngine, PencilBeamSource, VoxelGrid

    grid = VoxelGrid.uniform_water((12, 12, 12), (0.5, 0.5, 0.5))
    xs = AnalyticCrossSections(geometry_densities=grid.max_density_by_material())
    engine = HipEngine(grid, xs if rows == 1 else TwoEqualRows(xs), queue_factor=64)
    source = PencilBeamSource(energy, (3.0, 3.0, 0.01), (0.0, 0.0, 1.0))
    options = dict(primary_kind=kind, msc_model="gaussian", ecut=ecut, pcut=0.05, seed=4)
    engine._ctx.call("hmc_set_round_stacks", 0, 0)
    none = engine.run(source, histories, 2, **options)
    assert none.counters["trapped"] == 0
    assert none.counters["electron_pushes"] > (20 * histories if kind == "electron" else histories // 10)
    rounds = {}
    for slots in ((32, 32), (1, 1), (3, 5), (32, 0), (0, 32)):
        engine._ctx.call("hmc_set_round_stacks", *slots)
        got = engine.run(source, histories, 2, **options)
        _same(none, got)
        for name in ("electron_pushes", "electron_pops", "photon_pushes", "photon_pops"):
            assert got.counters[name] == none.counters[name], (slots, name)
        rounds[slots] = got.counters["rounds"]
    if kind == "electron":  # delta electrons that stay with their wave need no further round
        assert rounds[(32, 32)] < none.counters["rounds"] == rounds[(32, 0)]
    for bad in ((-1, 0), (0, 33)):
        with pytest.raises(ValueError):
            engine._ctx.call("hmc_set_round_stacks", *bad)
    engine.close()


def test_chunks_of_few_electrons_equal_one_chunk():
    """Whole waves of electrons whose stacks fill, against chunks of eight that hold a wave
    to a few particles."""
    from pyradmc_amd import AnalyticCrossSections, HipEngine, PencilBeamSource, VoxelGrid

    grid = VoxelGrid.uniform_water((12, 12, 12), (0.5, 0.5, 0.5))
    xs = AnalyticCrossSections(geometry_densities=grid.max_density_by_material())
    source = PencilBeamSource(6.0, (3.0, 3.0, 0.01), (0.0, 0.0, 1.0))
    options = dict(primary_kind="electron", msc_model="gaussian", ecut=0.02, pcut=0.01, seed=4)
    full = HipEngine(grid, xs, queue_factor=64).run(source, 512, 2, **options)
    few = HipEngine(grid, xs, chunk_size=8, queue_factor=512).run(source, 512, 2, **options)
    _same(full, few)
    pushed = full.counters["electron_pushes"]
    assert pushed > 4 * 512  # several delta electrons per primary


@pytest.mark.parametrize("columns, slots, blocks", [(1, 1, 1), (3, 7, 1), (2, 6, 2), (5, 3, 3), (1, 0, 1)])
def test_folds_in_one_pass_equal_their_parts(columns, slots, blocks):
    """Random quanta through hmc_fold_finalize (the first fold, a later one, the only one)
    and hmc_truncate against numpy's float64, bit for bit; a run with nothing folded."""
    from pyradmc_amd import _native as nat

    rng = np.random.default_rng(columns + slots)
    shape = (5, 7, 29)  # 1015 voxels: a remainder in every chunk
    n_vox = int(np.prod(shape))
    mass = rng.uniform(0.1, 2.0, n_vox)
    mass[::97] = 0.0
    ctx = nat.Context(0)
    zero, one = np.zeros(3), np.ones(3)
    ctx.call("hmc_set_scoring", *shape, nat.ptr(zero, nat.c_double), nat.ptr(one, nat.c_double),
             nat.ptr(mass, nat.c_double), columns, max(slots, 1))
    mean, sigma = np.empty((columns, n_vox)), np.empty((columns, n_vox))
    n_batches = max(slots * blocks, 1)
    s1, s2 = np.zeros((columns, n_vox)), np.zeros((columns, n_vox))
    total = 0
    for block in range(blocks if slots else 0):
        quanta = rng.integers(0, 10**9, (slots, columns, n_vox)) * (rng.random((slots, columns, n_vox)) < 0.2)
        quanta = np.ascontiguousarray(quanta, dtype=np.int64)
        nhist = np.ascontiguousarray(rng.integers(1, 1000, (slots, columns)), dtype=np.float64)
        ctx.call("hmc_set_quanta", nat.ptr(quanta, nat.c_int64))
        if block + 1 < blocks:
            ctx.call("hmc_fold", slots, nat.ptr(nhist, nat.c_double), None)
        else:
            ctx.call("hmc_fold_finalize", slots, nat.ptr(nhist, nat.c_double), n_batches, nat.ptr(mean, nat.c_double),
                     nat.ptr(sigma, nat.c_double))
        total += int(quanta.sum())
        for q, n in zip(quanta, nhist):
            with np.errstate(divide="ignore", invalid="ignore"):
                d = np.where(mass > 0.0, q * 1.0e-9 / (mass * n[:, None]), 0.0)
            s1, s2 = s1 + d, s2 + d * d
    if not slots:
        ctx.call("hmc_finalize", n_batches, nat.ptr(mean, nat.c_double), nat.ptr(sigma, nat.c_double))
    want = s1 / n_batches
    var = np.maximum(0.0, s2 / n_batches - want * want) * n_batches / max(n_batches - 1.0, 1.0)
    np.testing.assert_array_equal(mean, want)
    np.testing.assert_array_equal(sigma, np.sqrt(var / n_batches) if n_batches > 1 else np.zeros_like(want))
    folded, kept, entries = nat.c_int64(), np.zeros(columns, np.int64), nat.c_int64()
    ctx.call("hmc_folded_quanta", nat.ctypes.byref(folded))
    assert folded.value == total
    ctx.call("hmc_truncate", 0.3, nat.ptr(kept, nat.c_int64), nat.ctypes.byref(entries))
    expected = (want > 0.0) & (want >= 0.3 * want.max(axis=1, keepdims=True))
    np.testing.assert_array_equal(kept, expected.sum(axis=1))
    ctx.close()


def test_a_fold_after_the_finalize_renews_the_column_maxima():
    """hmc_truncate against the sums as they stand: a fold that follows the last one raises
    one column's largest value, so the threshold moves with it."""
    from pyradmc_amd import _native as nat

    n_vox, columns = 300, 2
    ctx = nat.Context(0)
    zero, one, mass = np.zeros(3), np.ones(3), np.ones(n_vox)
    ctx.call("hmc_set_scoring", n_vox, 1, 1, nat.ptr(zero, nat.c_double), nat.ptr(one, nat.c_double),
             nat.ptr(mass, nat.c_double), columns, 1)
    first = np.tile(np.arange(1, n_vox + 1, dtype=np.int64) * 10**9, (1, columns, 1))
    later = np.zeros_like(first)
    later[0, 1, 7] = 10**13
    nhist = np.ones((1, columns))
    kept, entries = np.zeros(columns, np.int64), nat.c_int64()

    def truncated():
        ctx.call("hmc_truncate", 0.5, nat.ptr(kept, nat.c_int64), nat.ctypes.byref(entries))
        return kept.tolist()

    ctx.call("hmc_set_quanta", nat.ptr(first, nat.c_int64))
    ctx.call("hmc_fold_finalize", 1, nat.ptr(nhist, nat.c_double), 1, None, None)
    assert truncated() == [n_vox // 2 + 1] * 2
    for fold in (("hmc_fold", 1, nat.ptr(nhist, nat.c_double), None),
                 ("hmc_fold_finalize", 1, nat.ptr(nhist, nat.c_double), 1, None, None)):
        ctx.call("hmc_set_quanta", nat.ptr(later, nat.c_int64))
        ctx.call(*fold)
        assert truncated() == [n_vox // 2 + 1, 1]
    ctx.close()


def test_a_grid_that_could_not_be_set_is_not_used():
    """After hmc_set_gs has failed (here for want of memory), no transport reads what is
    left of the cells before it; the next run uploads tables and grid again."""
    from pyradmc_amd import AnalyticCrossSections, HipEngine, PencilBeamSource, VoxelGrid
    from pyradmc_amd import _native as nat

    grid = VoxelGrid.uniform_water((8, 8, 8), (1.0, 1.0, 1.0))
    eng = HipEngine(grid, AnalyticCrossSections(geometry_densities=grid.max_density_by_material()))
    source = PencilBeamSource(6.0, (4.0, 4.0, -1.0), (0.0, 0.0, 1.0))
    before = eng.run(source, 1000, 2, seed=1)
    nodes = np.zeros(8, np.float32)
    with pytest.raises(MemoryError):
        eng._ctx.call("hmc_set_gs", nat.ptr(nodes, nat.ctypes.c_float), 20_000, 20_000, 20_000, 0, 0)
    with pytest.raises(RuntimeError, match="GS grid not set"):
        eng.run(source, 1000, 2, seed=1)
    eng._uploaded_tables = None
    _same(before, eng.run(source, 1000, 2, seed=1))
    eng.close()
