"""Launch shape and HIP graphs: groups of four transport rounds replayed from a captured
graph, the lanes per CU of each round and the refill block change no bit of a result.
Graph replays are checked one by one against eager runs, with eager work and host
synchronisation between them, and with other work items (seeds) reusing the graph."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def slab():
    from pyradmc_amd import workloads

    grid, xs, src, _ = workloads.slab_phantom()
    return grid, xs, src


def _engine(grid, xs, **launch):
    from pyradmc_amd import HipEngine

    eng = HipEngine(grid, xs)
    if launch:
        eng.set_launch(**launch)
    return eng


def _same(a, b) -> None:
    np.testing.assert_array_equal(a.dose, b.dose)
    np.testing.assert_array_equal(a.dose_sigma, b.dose_sigma)
    for name in ("energy_emitted", "energy_deposited", "energy_escaped", "energy_unscored"):
        assert getattr(a, name) == getattr(b, name), name


def test_launch_shape_and_graphs_change_no_bit(slab):
    grid, xs, src = slab
    eager = _engine(grid, xs, use_graphs=False).run(src, 300_000, 4, seed=11)
    assert eager.counters["graph_launches"] == 0
    for launch in ({}, {"round_lanes_per_cu": 1024}, {"round_lanes_per_cu": 4096, "refill_block": 256},
                   {"refill_block": 128, "use_graphs": False}, {"round_lanes_per_cu": 1024, "push_chunk": 256},
                   {"refill_block": 512, "push_chunk": 128, "use_graphs": False}):
        got = _engine(grid, xs, **launch).run(src, 300_000, 4, seed=11)
        _same(eager, got)
        assert (got.counters["graph_launches"] > 0) == launch.get("use_graphs", True), launch


@pytest.mark.parametrize("histories", (63, 65, 12_345, 700_001, 3_000_000))
def test_rounds_sized_by_their_queue_match_a_fixed_shape(slab, histories):
    """An engine without set_launch sizes refill blocks, push chunks and the grid by the
    queue: less than a wave's worth, around one wave, and long enough for long blocks."""
    grid, xs, src = slab
    sized = _engine(grid, xs).run(src, histories, 1, seed=5)
    _same(_engine(grid, xs, round_lanes_per_cu=2048, refill_block=64, push_chunk=64).run(src, histories, 1, seed=5),
          sized)


def _round_grid(engine, histories):
    from pyradmc_amd import _native as nat

    got = (nat.c_int * 4)()
    engine._ctx.call("hmc_round_grid", int(histories), got)
    return dict(zip(("workgroups", "threads", "refill_block", "push_chunk"), got))


def test_knobs_left_out_stay_automatic(slab):
    """Setting one knob leaves the others to the queue's length, and set_launch() with
    nothing set gives back an engine on which it was never called."""
    grid, xs, src = slab
    eng = _engine(grid, xs)
    ref = eng.run(src, 300_000, 4, seed=11)
    fresh = eng.launch
    assert fresh == {"round_lanes_per_cu": 0, "refill_block": 0, "push_chunk": 0, "use_graphs": True}
    sized = _round_grid(eng, 300_000)
    eng.set_launch(use_graphs=False)
    assert eng.launch == {**fresh, "use_graphs": False} and _round_grid(eng, 300_000) == sized
    _same(ref, eng.run(src, 300_000, 4, seed=11))
    eng.set_launch(refill_block=128)
    assert eng.launch == {**fresh, "refill_block": 128}
    assert _round_grid(eng, 300_000) == {**sized, "refill_block": 128}
    _same(ref, eng.run(src, 300_000, 4, seed=11))
    eng.set_launch()
    assert eng.launch == fresh and _round_grid(eng, 300_000) == sized
    _same(ref, eng.run(src, 300_000, 4, seed=11))


@pytest.mark.parametrize("lanes", (0, 256, 512, 2048, 8192))
def test_round_grids_fill_the_cus_and_no_more(slab, lanes):
    """One material: a workgroup fills its CU, so a round has one to a CU at any width and
    number of histories. Two: 256-lane workgroups, as many as the width says, and by the
    histories (at least one to a CU) where none is set."""
    from tests.test_round_builds_gpu import TwoEqualRows

    grid, xs, src = slab
    one, two = _engine(grid, xs), _engine(grid, TwoEqualRows(xs))
    cus = one._info["cu_count"]
    for eng in (one, two):
        eng.set_launch(round_lanes_per_cu=lanes)
        eng.run(src, 1000, 1, seed=1)  # uploads the tables
    for histories in (1, 1000, 80_000, 10_000_000):
        got = _round_grid(one, histories)
        assert (got["workgroups"], got["threads"]) == (cus, 768)
        auto = min(3 * cus, max(cus, -(-histories // 256)))
        got = _round_grid(two, histories)
        assert (got["workgroups"], got["threads"]) == (lanes // 256 * cus if lanes else auto, 256)


def test_graph_replays_match_eager_runs(slab):
    grid, xs, src = slab
    eng = _engine(grid, xs)
    ref = _engine(grid, xs, use_graphs=False)
    expected = {seed: ref.run(src, 200_000, 2, seed=seed) for seed in (1, 2)}
    for seed in (1, 2, 1, 1, 2):  # replays of one captured graph across runs and seeds
        got = eng.run(src, 200_000, 2, seed=seed)
        assert got.counters["graph_launches"] > 0
        _same(expected[seed], got)
        _same(expected[seed], ref.run(src, 200_000, 2, seed=seed))  # eager work between replays


def test_profiled_runs_launch_one_by_one_between_graph_replays(slab):
    grid, xs, src = slab
    eng = _engine(grid, xs)
    plain = eng.run(src, 200_000, 2, seed=3)
    assert plain.counters["graph_launches"] > 0
    eng.set_profiling(True)
    timed = eng.run(src, 200_000, 2, seed=3)
    eng.set_profiling(False)
    _same(plain, timed)
    assert timed.counters["graph_launches"] == 0
    assert timed.counters["photon_kernel_ms"] > 0.0 and timed.counters["electron_kernel_ms"] > 0.0
    again = eng.run(src, 200_000, 2, seed=3)
    assert again.counters["graph_launches"] > 0
    _same(plain, again)


def test_launch_arguments_rejected(slab):
    grid, xs, _ = slab
    eng = _engine(grid, xs)
    for bad in ({"round_lanes_per_cu": 100}, {"round_lanes_per_cu": 16384}, {"refill_block": 96},
                {"refill_block": 2048}, {"push_chunk": 32}, {"push_chunk": 100}):
        with pytest.raises(ValueError):
            eng.set_launch(**bad)


def test_autotune_picks_a_shape_that_changes_no_bit(slab, tmp_path, monkeypatch):
    from pyradmc_amd import autotune

    monkeypatch.setenv("PYRADMC_AMD_CACHE", str(tmp_path / "autotune.json"))
    grid, xs, src = slab
    eng = _engine(grid, xs)
    candidates = {"round_lanes_per_cu": (1024, 2048), "refill_block": (64, 128), "chunk_size": (None, 100_000)}
    config = eng.autotune(src, 200_000, 2, seed=1, repeats=1, candidates=candidates)
    assert (tmp_path / "autotune.json").is_file()
    assert eng.launch["round_lanes_per_cu"] == config.round_lanes_per_cu
    again = _engine(grid, xs)
    assert again.autotune(src, 200_000, 2, seed=1) == config  # from the cache
    _same(_engine(grid, xs, use_graphs=False).run(src, 200_000, 2, seed=9), eng.run(src, 200_000, 2, seed=9))


def test_dij_autotune_picks_a_shape_that_changes_no_bit(tmp_path, monkeypatch):
    from pyradmc_amd import BeamletGridSource, VoxelGrid
    from pyradmc_amd.data.analytic import AnalyticCrossSections

    monkeypatch.setenv("PYRADMC_AMD_CACHE", str(tmp_path / "autotune.json"))
    grid = VoxelGrid.uniform_water((12, 12, 20), (0.5, 0.5, 0.5))
    xs = AnalyticCrossSections(geometry_densities=grid.max_density_by_material())
    src = BeamletGridSource(4.0, -0.1, (1.0, 5.0), (1.0, 5.0), 3, 3)
    eng = _engine(grid, xs)
    candidates = {"round_lanes_per_cu": (512, 1024), "push_chunk": (64, 256), "chunk_size": (None, 50_000)}
    config = eng.autotune_dij(src, 20_000, 4, seed=1, repeats=1, candidates=candidates, truncation=1e-3,
                              value_dtype=np.float32)
    assert "dij|" in (tmp_path / "autotune.json").read_text()
    assert eng.launch["round_lanes_per_cu"] == config.round_lanes_per_cu
    tuned = eng.run_dij(src, 20_000, 4, seed=5, truncation=1e-3)
    plain = _engine(grid, xs, use_graphs=False).run_dij(src, 20_000, 4, seed=5, truncation=1e-3)
    for name in ("indptr", "indices", "dose", "sigma"):
        np.testing.assert_array_equal(getattr(tuned, name), getattr(plain, name))
