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


def test_moller_stack_in_use_and_full_equals_one_never_used():
    """Electrons far above a low cutoff meet a Moller interaction in many lanes of a pass:
    a wave's stack fills and lanes wait in place. Chunks of eight histories hold the wave
    to a few particles, so nothing waits long."""
    from pyradmc_amd import AnalyticCrossSections, HipEngine, PencilBeamSource, VoxelGrid

    grid = VoxelGrid.uniform_water((12, 12, 12), (0.5, 0.5, 0.5))
    xs = AnalyticCrossSections(geometry_densities=grid.max_density_by_material())
    source = PencilBeamSource(6.0, (3.0, 3.0, 0.01), (0.0, 0.0, 1.0))
    options = dict(primary_kind="electron", msc_model="gaussian", ecut=0.02, pcut=0.01, seed=4)
    full = HipEngine(grid, xs, queue_factor=64).run(source, 512, 2, **options)
    few = HipEngine(grid, xs, chunk_size=8, queue_factor=512).run(source, 512, 2, **options)
    _same(full, few)
    pushed = full.counters["electron_pushes"]
    assert pushed > 64 * 512 // 16  # delta electrons by the dozen per primary
