"""The measured work of this package, as a user's program has it done.

Seven kinds of work, each through public entry points:

* ``run``      ``HipEngine.run``: dose and sigma of an open field on a voxel grid;
* ``dij``      ``HipEngine.run_dij``: a beamlet-resolved dose matrix (CSC);
* ``product``  ``DeviceDij.apply_device``: doses of many weight vectors at once;
* ``plan``     ``study.objective_and_gradient``: one evaluation of a fluence optimiser;
* ``predict``  ``Conv3dDenoiser.predict_tensor``: denoised windows (inference);
* ``train``    forward, loss, backward and optimiser step of the denoiser;
* ``head``     ``presolve_head`` into a resident phase space and the field it gives.

Transport results are integer tallies of particles that each carry their own random
stream, so they are the same bits for a seed under any schedule: those cases compare
exactly. Engines run at their default launch shape, as a program that never tunes does.
"""

from __future__ import annotations

import math
import warnings
from functools import lru_cache
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch

from pyradmc_amd import denoise  # before any engine: the denoiser runs on torch's HIP runtime
from pyradmc_amd import (
    MLC,
    AirColumn,
    AnalyticCrossSections,
    BeamFrame,
    BeamLimitingStack,
    CollimatedSource,
    DeviceDij,
    GaussianSpotBeamSource,
    HipEngine,
    JawPair,
    PencilBeamSource,
    ScoringGrid,
    SpectralBeamletSource,
    SpectralBeamSource,
    SpectralParallelBeamSource,
    VoxelGrid,
    bremsstrahlung_6mv_like,
    presolve_head,
    study,
    workloads,
)

MODEL = Path(denoise.__file__).resolve().parent / "models" / "denoiser_ct.npz"
SLOPE = 0.1  # the network's leaky ReLU
# Arithmetic of one history, for work(): about 11 electron steps and 2.6 photon steps
# on the 6 MV-like workloads; without electrons only the photon steps remain.
FLOPS_PER_HISTORY = {True: 2400, False: 250}

# A population smaller than the histories drawn from it is what a small field has.
warnings.filterwarnings("ignore", message=".*population.*")


# ----------------------------------------------------------------------- the cases


def listed():
    return [
        # The quick start: a pencil in a small water cube. Latency and launches.
        dict(name="pencil_quickstart", kind="run", nx=16, ny=16, nz=16, spacing=1.0, phantom="water",
             source="pencil", histories=80_000, batches=10, electrons=True, msc="gs", resolution=0.0, scoring="grid"),
        # The heterogeneous slab benchmark at its full statistics.
        dict(name="slab_field", kind="run", nx=64, ny=64, nz=96, spacing=0.2, phantom="slab", source="parallel",
             histories=10_000_000, batches=20, electrons=True, msc="gs", resolution=0.0, scoring="grid"),
        # A ragged CT-like volume under a diverging field with the other options in use:
        # Gaussian scattering, deposits spread along the step, a coarser dose grid.
        dict(name="ct_field_options", kind="run", nx=87, ny=61, nz=73, spacing=0.3, phantom="ct", source="fan",
             histories=2_000_000, batches=10, electrons=True, msc="gaussian", resolution=0.1, scoring="coarse"),
        # A jaw- and leaf-shaped field from a head pre-solved on the device.
        dict(name="head_field", kind="head", n=64, spacing=0.5, primaries=2_000_000, histories=2_000_000, batches=10),
        # The batched Dij: 100 beamlets with uneven counts on a CT-like volume.
        dict(name="dij_ct_uneven", kind="dij", nx=128, ny=128, nz=96, spacing=0.25, side=10, width=0.5, pitch=1.0,
             gantry=0.0, per_beamlet=200_000, uneven=True, batches=10, correlated=True, f32=False),
        # Part of one beam of the large plan, from an oblique gantry angle, float32 values.
        dict(name="dij_plan_beam", kind="dij", nx=256, ny=256, nz=128, spacing=0.2, side=6, width=0.5, pitch=0.5,
             gantry=72.0, per_beamlet=240_000, uneven=False, batches=10, correlated=True, f32=True),
        # Planning products: scenarios or robust-optimisation vectors over one beam's matrix.
        dict(name="product_f64", kind="product", nx=128, ny=128, nz=96, side=15, n_w=256, values="f64",
             precision="f64"),
        dict(name="product_f32", kind="product", nx=128, ny=128, nz=96, side=15, n_w=1000, values="f32",
             precision="f32"),
        # One evaluation inside a fluence optimisation: a product and a transpose product.
        dict(name="plan_step", kind="plan", nx=128, ny=128, nz=96, side=15, radius=12),
        # Denoising a batch of beamlet columns, and one training step on four crops.
        dict(name="denoise_batch", kind="predict", n=32, depth=96),
        dict(name="train_step", kind="train", n=4, depth=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("run", "run", "run", "dij", "dij", "product", "product", "product", "plan", "predict",
                       "predict", "train", "train", "head"))
    if kind == "run":
        source = rng.choice(("pencil", "parallel", "parallel", "fan"))
        nx, ny, nz = (rng.randint(15, 110) for _ in range(3))
        batches = rng.choice((1, 5, 10, 20))
        plain = rng.random() < 0.6
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, spacing=rng.choice((0.2, 0.25, 0.3, 0.5)),
                    phantom=rng.choice(("water", "slab", "ct")), source=source,
                    histories=batches * _log_int(rng, 20_000 / batches, 8_000_000 / batches), batches=batches,
                    electrons=rng.random() < 0.85, msc="gs" if plain else rng.choice(("gs", "gaussian")),
                    resolution=0.0 if plain else rng.choice((0.0, 0.05, 0.1)),
                    scoring="grid" if plain else rng.choice(("grid", "coarse")))
    if kind == "dij":
        nx, ny, nz = rng.randint(50, 140), rng.randint(50, 140), rng.randint(40, 110)
        side, batches = rng.randint(1, 9), rng.choice((1, 5, 10))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, spacing=rng.choice((0.2, 0.25, 0.3)), side=side,
                    width=rng.choice((0.3, 0.5)), pitch=0.5, gantry=rng.choice((0.0, 0.0, 72.0, 144.0)),
                    per_beamlet=batches * _log_int(rng, 2_000 / batches, 200_000 / batches),
                    uneven=rng.random() < 0.5, batches=batches, correlated=rng.random() < 0.7,
                    f32=rng.random() < 0.5)
    if kind == "product":
        nx, ny, nz = rng.randint(40, 128), rng.randint(40, 128), rng.randint(33, 96)
        precision = rng.choice(("f64", "f32"))
        most = 900 if precision == "f32" else 450
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, side=rng.randint(4, 15), n_w=_log_int(rng, 1, most),
                    values=rng.choice(("f64", "f32")), precision=precision)
    if kind == "plan":
        return dict(kind=kind, nx=rng.randint(60, 128), ny=rng.randint(60, 128), nz=rng.randint(40, 96),
                    side=rng.randint(4, 15), radius=rng.randint(4, 14))
    if kind == "predict":
        return dict(kind=kind, n=_log_int(rng, 1, 31), depth=8 * rng.randint(5, 13))
    if kind == "train":
        return dict(kind=kind, n=rng.randint(1, 6), depth=8 * rng.randint(4, 9))
    histories = 10 * _log_int(rng, 10_000, 200_000)
    return dict(kind=kind, n=rng.randint(30, 70), spacing=0.5, primaries=_log_int(rng, 100_000, 2_000_000),
                histories=histories, batches=10)


# ------------------------------------------------------------------------ transport


@lru_cache(maxsize=8)
def _grid(nx, ny, nz, spacing, phantom):
    """The phantoms of the package's workloads at any size: the voxels a program loads once."""
    shape = (nx, ny, nz)
    if phantom == "ct":
        return workloads.ct_like_grid(shape=shape, spacing=spacing)
    density = np.ones(shape)
    if phantom == "slab":  # lung from 16 % to 36 % of the depth, bone from 47 % to 57 %
        density[:, :, int(0.16 * nz):int(0.36 * nz)] = 0.26
        density[:, :, int(0.47 * nz):int(0.57 * nz)] = 1.85
    return VoxelGrid(shape=shape, spacing=(spacing,) * 3, density=density, material=np.zeros(shape, dtype=np.int32))


def _engine(grid):
    xs = AnalyticCrossSections(geometry_densities=grid.max_density_by_material())
    return HipEngine(grid, xs), xs


def _open_source(case):
    lx, ly, lz = (case[k] * case["spacing"] for k in ("nx", "ny", "nz"))
    if case["source"] == "pencil":
        return PencilBeamSource(6.0, (lx / 2, ly / 2, -1.0), (0.0, 0.0, 1.0))
    if case["source"] == "parallel":  # the middle of the face, up to 10 x 10 cm
        hx, hy = min(5.0, 0.4 * lx), min(5.0, 0.4 * ly)
        return SpectralParallelBeamSource(bremsstrahlung_6mv_like(), -0.1, (lx / 2 - hx, lx / 2 + hx),
                                          (ly / 2 - hy, ly / 2 + hy))
    side = min(8.0, 0.6 * min(lx, ly))
    return SpectralBeamSource(bremsstrahlung_6mv_like(), (lx / 2, ly / 2, lz / 2 - 100.0), (lx / 2, ly / 2, lz / 2),
                              side, side)


def _prepare_run(case, seed):
    grid = _grid(case["nx"], case["ny"], case["nz"], case["spacing"], case["phantom"])
    engine, _ = _engine(grid)
    scoring = None
    if case["scoring"] == "coarse":  # voxels half again as wide, over the middle of the grid
        shape = tuple(max(1, int(n / 1.6)) for n in grid.shape)
        wide = 1.5 * case["spacing"]
        origin = tuple((n * case["spacing"] - m * wide) / 2 for n, m in zip(grid.shape, shape))
        scoring = ScoringGrid.rebin(grid, shape, (wide,) * 3, origin)
    options = dict(transport_electrons=case["electrons"], msc_model=case["msc"], scoring_grid=scoring,
                   deposit_resolution_cm=case["resolution"] or None)
    return SimpleNamespace(engine=engine, source=_open_source(case), histories=case["histories"],
                           batches=case["batches"], seed=seed, options=options)


def _dose(r):
    return {"dose": r.dose, "sigma": r.dose_sigma, "emitted": r.energy_emitted, "deposited": r.energy_deposited,
            "escaped": r.energy_escaped, "unscored": r.energy_unscored}


def _run_run(s):
    return _dose(s.engine.run(s.source, s.histories, s.batches, seed=s.seed, **s.options))


def _prepare_dij(case, seed):
    grid = _grid(case["nx"], case["ny"], case["nz"], case["spacing"], "ct")
    engine, _ = _engine(grid)
    iso = np.array([n * case["spacing"] / 2 for n in grid.shape])
    t = math.radians(case["gantry"])
    d, u, v = (np.array(a) for a in ((math.sin(t), 0.0, math.cos(t)), (math.cos(t), 0.0, -math.sin(t)),
                                     (0.0, 1.0, 0.0)))
    half = (case["side"] - 1) / 2
    centers = [tuple(iso + (i - half) * case["pitch"] * u + (j - half) * case["pitch"] * v)
               for i in range(case["side"]) for j in range(case["side"])]
    source = SpectralBeamletSource(bremsstrahlung_6mv_like(), tuple(iso - 100.0 * d), centers, case["width"],
                                   case["width"], u_axis=tuple(u), v_axis=tuple(v))
    counts = case["per_beamlet"]
    if case["uneven"]:
        counts = workloads.lognormal_counts(len(centers), case["batches"], median=counts)
    value = np.float32 if case["f32"] else np.float64
    options = dict(truncation=1e-4, correlated=case["correlated"], value_dtype=value)
    # A seed's matrix has its own number of entries. The outputs have the same shape for
    # every seed: the entries up to `fixed`, as the engine returned them, and the few
    # beyond it in kept arrays of `slack` entries, both sized by a run of a fixed seed.
    entries = engine.run_dij(source, counts, case["batches"], seed=17, **options).indices.size
    spread = 0.01 + min(0.4, 30.0 / math.sqrt(entries))
    fixed, slack = int((1 - spread) * entries), int(2 * spread * entries) + 64
    rest = {"indices": np.zeros(slack, np.int64), "dose": np.zeros(slack, value), "sigma": np.zeros(slack, value)}
    return SimpleNamespace(engine=engine, source=source, counts=counts, batches=case["batches"], seed=seed,
                           options=options, fixed=fixed, rest=rest)


def _run_dij(s):
    r = s.engine.run_dij(s.source, s.counts, s.batches, seed=s.seed, **s.options)
    out = {"indptr": r.indptr, "emitted": r.energy_emitted, "deposited": r.energy_deposited,
           "escaped": r.energy_escaped}
    for name, rest in s.rest.items():
        a = getattr(r, name)
        beyond = a.size - s.fixed
        if 0 <= beyond <= rest.size:
            rest[:beyond], rest[beyond:] = a[s.fixed:], 0
            out[name], out[name + "_rest"] = a[:s.fixed], rest
        else:
            out[name] = a
    return out


def _prepare_head(case, seed):
    """Two focused jaw pairs and a 40-pair rounded-tip MLC over a water cube; the
    analytic data is water only, so the devices are water at tungsten's density."""
    n, spacing = case["n"], case["spacing"]
    grid = _grid(n, n, n, spacing, "water")
    engine, xs = _engine(grid)
    c = n * spacing / 2
    focal = (c, c, -100.0)
    leaves = np.linspace(-2.0, 2.0, 41)
    mid = 0.5 * (leaves[:-1] + leaves[1:])
    stack = BeamLimitingStack(BeamFrame(focal), (
        JawPair("v", 20.0, 27.8, -2.2, 2.2, 0, 19.3, focused=True),
        JawPair("u", 28.0, 35.8, -2.2, 2.2, 0, 19.3, focused=True),
        MLC(40.0, 46.5, tuple(leaves), tuple(-1.2 - 0.6 * np.cos(mid)), tuple(0.9 + 0.7 * np.sin(mid) ** 2), 8.0, 0,
            18.0, focused_sides=True),
    ))
    spot = GaussianSpotBeamSource(bremsstrahlung_6mv_like(), focal, (c, c, -85.0), 3.0, 3.0, 0.15, 0.15)
    head = dict(cross_sections=xs, exit_z=97.0, stack=stack, air=AirColumn(50.0, 95.0, material=0), engine=engine,
                resident=True)
    return SimpleNamespace(engine=engine, spot=spot, head=head, collimated=CollimatedSource(spot, stack, xs),
                           primaries=case["primaries"], histories=case["histories"], batches=case["batches"],
                           seed=seed)


def _run_head(s):
    """The pre-solve, the field it gives, and the same field collimated in the generator."""
    population = presolve_head(s.spot, n_histories=s.primaries, seed=s.seed, **s.head)
    field = s.engine.run(population, s.histories, s.batches, seed=s.seed + 1)
    shaped = s.engine.run(s.collimated, s.histories, s.batches, seed=s.seed + 2)
    return {"particles": len(population), "field": _dose(field), "shaped": _dose(shaped)}


# ------------------------------------------------------------------ planning products


def _beam_matrix(nx, ny, nz, side, seed):
    """A CSC like one beam's truncated Dij: per beamlet a core along z of about 2 voxels
    radius and a scatter tail that Monte Carlo noise keeps or drops voxel by voxel.
    (indptr, indices, values), float64, on the GPU."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    x = torch.arange(nx, device=dev, dtype=torch.float32)[:, None]
    y = torch.arange(ny, device=dev, dtype=torch.float32)[None, :]
    depth = torch.exp(-0.012 * torch.arange(nz, device=dev, dtype=torch.float32))
    indptr, indices, values = [0], [], []
    for j in range(side * side):
        cx = nx / 2 + 2.5 * (j // side - (side - 1) / 2)
        cy = ny / 2 + 2.5 * (j % side - (side - 1) / 2)
        r = torch.sqrt((x - cx) ** 2 + (y - cy) ** 2)
        lateral = torch.sigmoid(3.0 * (1.4 - r)) + 0.01 * torch.exp(-r / 9.0)
        mean = (lateral[:, :, None] * depth).reshape(-1)
        keep = torch.rand(mean.numel(), generator=gen, device=dev) < (mean / 0.012).clamp(max=1.0)
        at = keep.nonzero().squeeze(1)
        noise = torch.rand(at.numel(), generator=gen, device=dev, dtype=torch.float64)
        indices.append(at)
        values.append(mean[at].double().clamp(min=2e-4) * (0.6 + 0.8 * noise))
        indptr.append(indptr[-1] + at.numel())
    return np.array(indptr, dtype=np.int64), torch.cat(indices), torch.cat(values)


def _weights(case, seed, columns):
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    return torch.rand(columns, generator=gen, device="cuda", dtype=torch.float64)


def _host_matrix(case, seed, dtype):
    indptr, indices, values = _beam_matrix(case["nx"], case["ny"], case["nz"], case["side"], seed)
    return SimpleNamespace(indptr=indptr, indices=indices.cpu().numpy(), dose=values.cpu().numpy().astype(dtype),
                           n_beamlets=case["side"] ** 2, grid_shape=(case["nx"], case["ny"], case["nz"]),
                           n_voxels=case["nx"] * case["ny"] * case["nz"])


def _np_dtype(name):
    return np.float64 if name == "f64" else np.float32


def _prepare_product(case, seed):
    dij = _host_matrix(case, seed, _np_dtype(case["values"]))
    dtype = torch.float64 if case["precision"] == "f64" else torch.float32
    w = _weights(case, seed, (dij.n_beamlets, case["n_w"])).to(dtype)
    return SimpleNamespace(dij=DeviceDij(dij), w=w,
                           out=torch.empty((dij.n_voxels, case["n_w"]), dtype=dtype, device="cuda"))


def _run_product(s):
    s.dij.apply_device(s.w, s.out)
    return s.out


def _exact_product(case, seed):
    indptr, rows, values = _beam_matrix(case["nx"], case["ny"], case["nz"], case["side"], seed)
    if case["values"] == "f32":
        values = values.float().double()
    n_cols, n_vox = case["side"] ** 2, case["nx"] * case["ny"] * case["nz"]
    w = _weights(case, seed, (n_cols, case["n_w"]))
    if case["precision"] == "f32":
        w = w.float().double()
    out = torch.zeros((n_vox, case["n_w"]), dtype=torch.float64, device="cuda")
    for j in range(n_cols):  # a column's rows are distinct
        lo, hi = int(indptr[j]), int(indptr[j + 1])
        out[rows[lo:hi]] += values[lo:hi, None] * w[j]
    return out


def _regions(case):
    """A spherical target in the middle of the volume and a box of healthy tissue beside it."""
    x, y, z = np.ogrid[:case["nx"], :case["ny"], :case["nz"]]
    cx, cy, cz, r = case["nx"] // 2, case["ny"] // 2, case["nz"] // 2, case["radius"]
    ptv = (x - cx) ** 2 + (y - cy) ** 2 + (z - cz) ** 2 <= r * r
    oar = (np.abs(x - cx - 2 * r) <= r // 2 + 1) & (np.abs(y - cy) <= r) & (np.abs(z - cz) <= r)
    return ptv.reshape(-1), (oar & ~ptv).reshape(-1)


def _prepare_plan(case, seed):
    ptv, oar = _regions(case)
    problem = study.ToyPlanProblem(_host_matrix(case, seed, np.float64), ptv, oar, prescription=2.0, oar_penalty=2.0)
    w = _weights(case, seed, (case["side"] ** 2,)).cpu().numpy() * 2.0
    study.objective_and_gradient(problem, w)  # the region's rows go to the device on the first evaluation
    return SimpleNamespace(problem=problem, w=w)


def _run_plan(s):
    f, gradient = study.objective_and_gradient(s.problem, s.w)
    return {"objective": f, "gradient": gradient}


def _exact_plan(case, seed):
    ptv, oar = _regions(case)
    dij = _host_matrix(case, seed, np.float64)
    w = _weights(case, seed, (case["side"] ** 2,)).cpu().numpy() * 2.0
    column = np.repeat(np.arange(dij.n_beamlets), np.diff(dij.indptr))
    d = np.bincount(dij.indices, weights=dij.dose * w[column], minlength=dij.n_voxels)
    a = np.zeros(dij.n_voxels)
    r = d[ptv] - 2.0
    f = float(r @ r) / r.size
    a[ptv] = 2.0 / r.size * r
    if oar.any():
        over = np.maximum(0.0, d[oar] - 0.3 * 2.0)
        f += 2.0 * float(over @ over) / over.size
        a[oar] += 2.0 * 2.0 / over.size * over
    return {"objective": f, "gradient": np.bincount(column, weights=dij.dose * a[dij.indices],
                                                    minlength=dij.n_beamlets)}


# ------------------------------------------------------------------------- denoiser


def _columns(n, depth, seed):
    """Scaled low-history beamlet columns, their full-statistics targets and densities,
    [n][depth][64][64] on the GPU (network axes)."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def rand(*shape):
        return torch.rand(shape, generator=gen, device=dev)

    z = torch.arange(depth, device=dev)[None, :, None, None] / 96.0
    c = torch.arange(64, device=dev, dtype=torch.float32) - 31.5
    dx, dy = (c[None, None, :, None] - 3.0 * rand(n, 1, 1, 1)), (c[None, None, None, :] - 3.0 * rand(n, 1, 1, 1))
    r = torch.sqrt(dx * dx + dy * dy)
    target = torch.exp(-1.1 * z) * (torch.sigmoid(2.5 * (1.6 - r)) + 0.02 * torch.exp(-r / 6.0))
    density = torch.where(r + 12.0 * rand(n, 1, 1, 1) < 30.0, 1.0, 0.05) * (0.3 + 1.4 * rand(n, depth // 8, 8, 8)
                                                                            .repeat_interleave(8, 1)
                                                                            .repeat_interleave(8, 2)
                                                                            .repeat_interleave(8, 3))
    spread = torch.sqrt(0.004 * target + 1e-7)
    noisy = (target + spread * torch.randn(target.shape, generator=gen, device=dev)).clamp(min=0.0)
    noisy = torch.where(rand(*target.shape) < (target / 2e-3).clamp(max=1.0), noisy, torch.zeros_like(noisy))
    return noisy, target.contiguous(), density


def _packed(noisy, density):
    """The network's input as the data pipeline leaves it on the device: 16 channels in
    bf16 (dose, half the density, zeros) and the channel-major copy."""
    return denoise.pack_input(noisy.cpu().numpy(), (0.5 * density).cpu().numpy())


def _prepare_predict(case, seed):
    noisy, _, density = _columns(case["n"], case["depth"], seed)
    x, _ = _packed(noisy, density)
    return SimpleNamespace(model=denoise.load(MODEL), x=x)


def _run_predict(s):
    return s.model.predict_tensor(s.x)


def _prepare_train(case, seed):
    noisy, target, density = _columns(case["n"], case["depth"], seed)
    x, x_cm = _packed(noisy, density)
    weight = target + 0.01
    return SimpleNamespace(model=denoise.load(MODEL), x=x, x_cm=x_cm, target=target, weight=weight / weight.mean())


def _run_train(s):
    out, cache = s.model.forward(s.x, s.x_cm, keep=True)
    partial, dout, dout_cm = s.model.loss_and_grad(out, s.x, s.target, s.weight, 1.0 / s.target.numel())
    s.model.backward(cache, dout, dout_cm)
    s.model.adam_step(1e-5)
    layers = s.model.layers
    # The biases' gradients are one output: a single one can cancel to almost nothing.
    return {"loss": partial.sum(), "b": torch.cat([lay.gb for lay in layers.values()]),
            **{name: lay.gw for name, lay in layers.items()}}


def _network(x, p):
    """The network in float64, [n][d][h][w][c], as autograd reads it."""

    def conv(t, name, activate=True):
        w, b = p[name + ".w"], p[name + ".b"]
        n, d, h, wd, _ = t.shape
        pad = torch.nn.functional.pad(t, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b.expand(n * d * h * wd, -1)
        for tap in range(27):
            z, yy, xx = tap // 9, tap // 3 % 3, tap % 3
            part = pad[:, z:z + d, yy:yy + h, xx:xx + wd, :].reshape(-1, t.shape[4])
            y = y + part @ w[tap].t().contiguous()
        y = y.reshape(n, d, h, wd, -1)
        return torch.where(y > 0, y, SLOPE * y) if activate else y

    def pool(t):
        n, d, h, w, c = t.shape
        return t.reshape(n, d // 2, 2, h // 2, 2, w // 2, 2, c).mean(dim=(2, 4, 6))

    def up(t):
        return t.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    s0 = conv(conv(x, "e0a"), "e0b")
    s1 = conv(conv(pool(s0), "e1a"), "e1b")
    s2 = conv(conv(pool(s1), "e2a"), "e2b")
    t = conv(conv(pool(s2), "e3a"), "e3b")
    t = conv(conv(up(t), "d2a") + s2, "d2b")
    t = conv(conv(up(t), "d1a") + s1, "d1b")
    t = conv(conv(up(t), "d0a") + s0, "d0b")
    return conv(t, "head", activate=False)[..., 0] + x[..., 0]


def _float64_inputs(noisy, density):
    x = torch.zeros(tuple(noisy.shape) + (16,), dtype=torch.float64, device="cuda")
    x[..., 0] = noisy.to(torch.bfloat16).double()
    x[..., 1] = (0.5 * density).to(torch.bfloat16).double()
    with np.load(MODEL, allow_pickle=False) as f:
        p = {k: torch.from_numpy(np.asarray(f[k], dtype=np.float64)).cuda() for k in f.files if k[-2:] in (".w", ".b")}
    return x, p


def _exact_predict(case, seed):
    noisy, _, density = _columns(case["n"], case["depth"], seed)
    x, p = _float64_inputs(noisy, density)
    with torch.no_grad():
        return torch.cat([_network(x[k:k + 4], p) for k in range(0, case["n"], 4)])


def _exact_train(case, seed):
    noisy, target, density = _columns(case["n"], case["depth"], seed)
    x, p = _float64_inputs(noisy, density)
    weight = target + 0.01
    weight = (weight / weight.mean()).double()
    total, grads = 0.0, {k: torch.zeros_like(v) for k, v in p.items()}
    for k in range(case["n"]):
        leaves = {name: v.clone().requires_grad_() for name, v in p.items()}
        pred = _network(x[k:k + 1], leaves)
        loss = (weight[k:k + 1] * (pred - target[k:k + 1].double()) ** 2).sum()
        (loss / target.numel()).backward()
        total += float(loss.detach())
        for name, v in leaves.items():
            grads[name] += v.grad
    names = [name for name, _, _ in denoise.layer_specs(denoise.CIN_PAD, (16, 32, 64, 128))]
    return {"loss": total, "b": torch.cat([grads[n + ".b"] for n in names]), **{n: grads[n + ".w"] for n in names}}


# ------------------------------------------------------------------------ interface

_PREPARE = dict(run=_prepare_run, dij=_prepare_dij, head=_prepare_head, product=_prepare_product, plan=_prepare_plan,
                predict=_prepare_predict, train=_prepare_train)
_RUN = dict(run=_run_run, dij=_run_dij, head=_run_head, product=_run_product, plan=_run_plan, predict=_run_predict,
            train=_run_train)
_EXACT = dict(product=_exact_product, plan=_exact_plan, predict=_exact_predict, train=_exact_train)


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state.kind = case["kind"]
    return state


def run(state):
    return _RUN[state.kind](state)


def exact(case, seed):
    """Monte Carlo doses have no value but the sampled one; the rest in float64."""
    make = _EXACT.get(case["kind"])
    return make(case, seed) if make else None


def work(case):
    kind = case["kind"]
    if kind in ("run", "dij"):
        voxels = case["nx"] * case["ny"] * case["nz"]
        if kind == "run":
            # density, material and mass in, dose and sigma out
            return {"bytes": 29 * voxels, "flops": FLOPS_PER_HISTORY[case["electrons"]] * case["histories"]}
        columns = case["side"] ** 2
        mean = math.exp(0.32) if case["uneven"] else 1.0  # lognormal counts, sigma 0.8
        kept = 0.06 * voxels * columns  # entries above the truncation, about
        return {"bytes": 13 * voxels + (16 if case["f32"] else 24) * kept,
                "flops": FLOPS_PER_HISTORY[True] * case["per_beamlet"] * mean * columns}
    if kind == "head":
        return {"bytes": 2 * 29 * case["n"] ** 3 + 36 * case["primaries"],
                "flops": 3000 * case["primaries"] + 2 * FLOPS_PER_HISTORY[True] * case["histories"]}
    if kind in ("product", "plan"):
        voxels, columns = case["nx"] * case["ny"] * case["nz"], case["side"] ** 2
        if kind == "plan":  # the region's share of the entries, read by each of the two products
            region = 6.0 * case["radius"] ** 3
            entries = 0.25 * region * columns
            return {"bytes": 2 * 12 * entries + 16 * region, "flops": 4 * entries}
        entries = 0.045 * voxels * columns
        value, out = (8 if case[k] == "f64" else 4 for k in ("values", "precision"))
        return {"bytes": (4 + value) * entries + out * case["n_w"] * (voxels + columns),
                "flops": 2 * entries * case["n_w"]}
    shape = (case["n"], case["depth"], 64, 64)
    flops = denoise.forward_flops(shape)
    voxels = case["n"] * case["depth"] * 64 * 64
    if kind == "predict":  # the packed input in, the prediction out
        return {"bytes": 36 * voxels, "flops": flops}
    weights = sum(27 * a * b for _, a, b in denoise.layer_specs(denoise.CIN_PAD, (16, 32, 64, 128)))
    # the packed input twice, target and weight in; masters, moments and gradients of the weights
    return {"bytes": 72 * voxels + 32 * weights, "flops": 3 * flops}


def tolerance(case):
    """About four times what each path is from float64, as measured: 9e-8 for float32
    products, 1.4e-15 for the optimiser's sums, 2.9e-3 for the bf16 network's output. Its
    weight gradients are 0.03 to 0.08 off (bf16 activations and gradients rounded in every
    layer, the deepest levels and the smallest batches worst); two roundings differ by
    about as much again."""
    kind = case["kind"]
    if kind in ("run", "dij", "head"):
        return "exact"
    if kind == "product":  # float64 products are the sequential float64 sum, bit for bit
        return "exact" if case["precision"] == "f64" else {"rel": 4e-7}
    if kind == "plan":
        return {"rel": 1e-14}
    return {"rel": 1.2e-2 if kind == "predict" else 0.12}
