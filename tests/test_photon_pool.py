"""The transport kernels keep photons of a wave in an LDS pool and run flights,
interactions and sampling when enough lanes can take part. Schedules never
change a history: every threshold, register budget, block size, staging of the
tables and bounds (which sets the pool's size) and run size gives the events of
the default run."""
import numpy as np
import pytest

from dxmclib_amd import backend, capi

pytestmark = pytest.mark.gpu

NAMES = ["Water, Liquid", "Bone, Cortical (ICRU)", "Lung (ICRU)", "Adipose Tissue (ICRP)"]
DENSITIES = [1.0, 1.92, 0.26, 0.95]


@pytest.mark.parametrize("n_materials", [1, 20, 40, 64])
@pytest.mark.parametrize("measured", [False, True])
def test_schedules_run_the_same_histories(device, n_materials, measured):
    rng = np.random.default_rng(6)
    shape = (45, 39, 43)
    names = (NAMES * 16)[:n_materials]
    mat = rng.integers(0, n_materials, shape).astype(np.uint8)
    dens = np.array((DENSITIES * 16)[:n_materials])[mat]
    if not measured:
        dens = dens * rng.uniform(0.95, 1.05, shape)
    meas = np.zeros(shape, np.uint8)
    meas[10:30, 10:30, 12:30] = 1
    spacing = (1.0, 1.3, 0.9)
    w = device.upload_world(mat, dens, spacing, backend.world_extent(shape[::-1], spacing), n_materials, meas if measured else None)
    tables = backend.HostTables(names, device.world_max_density(w, n_materials), 100.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=100.0, al_mm=2.5, sdd=1000.0, field_size=(60.0, 60.0), histories_per_exposure=1, total_exposures=3)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    settings = [dict(), dict(flags=capi.RUN_COUNTERS | capi.RUN_EXACT_STEPS), dict(waves_per_simd=4), dict(lds_tables=1), dict(lds_tables=3),
                dict(regeneration_threshold=1, interaction_threshold=1), dict(regeneration_threshold=64, interaction_threshold=64),
                dict(regeneration_threshold=1, interaction_threshold=64, queue_depth=64, blocks_per_cu=1), dict(histories_per_launch=777)]
    try:
        for model in (1, 2):
            for size in (1, 21, 22, 1500, 40_001):  # histories an exposure: below, at and above a wave's, and many waves
                for x in exposures:
                    x.n_histories = size
                ref = None
                for k in settings if size in (22, 40_001) else settings[:2]:
                    print(f"pool materials {n_materials} measured {measured} L={model} size {size} {k}", flush=True)
                    cfg = capi.RunCfg()
                    for f, v in k.items():
                        setattr(cfg, f, v)
                    tally = device.tally(mat.size)
                    stats = device.run(w, t, exposures, tally, capi.PRECISION_FP32, model, seed=29, tuning=cfg)
                    dose, events, _ = device.download(tally, mat.size)
                    device.destroy_tally(tally)
                    assert stats.histories == 3 * size and int(events.sum()) == stats.events
                    if ref is None:
                        ref = (stats.steps, stats.events, events, dose)
                        continue
                    assert (stats.steps, stats.events) == ref[:2]
                    assert np.array_equal(events, ref[2])
                    assert np.allclose(dose, ref[3], rtol=1e-10, atol=0)
    finally:
        device.destroy_tables(t)
        device.destroy_world(w)


# code worlds: bounds and tables in LDS, the tables alone (22 at L = 1), none
@pytest.mark.parametrize("n_materials", [1, 22, 64])
@pytest.mark.parametrize("measured", [False, True])
def test_fp64_schedules_run_the_same_histories(device, n_materials, measured):
    rng = np.random.default_rng(7)
    shape = (45, 39, 43)
    names = (NAMES * 16)[:n_materials]
    mat = rng.integers(0, n_materials, shape).astype(np.uint8)
    dens = np.array((DENSITIES * 16)[:n_materials])[mat]
    if not measured:
        dens = dens * rng.uniform(0.95, 1.05, shape)
    meas = np.zeros(shape, np.uint8)
    meas[10:30, 10:30, 12:30] = 1
    spacing = (1.0, 1.3, 0.9)
    w = device.upload_world(mat, dens, spacing, backend.world_extent(shape[::-1], spacing), n_materials, meas if measured else None)
    tables = backend.HostTables(names, device.world_max_density(w, n_materials), 100.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=100.0, al_mm=2.5, sdd=1000.0, field_size=(60.0, 60.0), histories_per_exposure=1, total_exposures=3)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    settings = [dict(), dict(flags=capi.RUN_COUNTERS | capi.RUN_EXACT_STEPS), dict(block_size=64), dict(block_size=192), dict(block_size=256),
                dict(regeneration_threshold=1, interaction_threshold=1), dict(regeneration_threshold=64, interaction_threshold=64),
                dict(regeneration_threshold=1, interaction_threshold=64, queue_depth=64, blocks_per_cu=1), dict(histories_per_launch=777)]
    try:
        for model in (1, 2):
            for size in (22, 20_001):
                for x in exposures:
                    x.n_histories = size
                ref = None
                for k in settings:
                    print(f"fp64 pool materials {n_materials} measured {measured} L={model} size {size} {k}", flush=True)
                    cfg = capi.RunCfg()
                    for f, v in k.items():
                        setattr(cfg, f, v)
                    tally = device.tally(mat.size)
                    stats = device.run(w, t, exposures, tally, capi.PRECISION_FP64, model, seed=29, tuning=cfg)
                    dose, events, _ = device.download(tally, mat.size)
                    device.destroy_tally(tally)
                    assert stats.histories == 3 * size and int(events.sum()) == stats.events
                    if ref is None:
                        ref = (stats.steps, stats.events, events, dose)
                        continue
                    assert (stats.steps, stats.events) == ref[:2]
                    assert np.array_equal(events, ref[2])
                    assert np.allclose(dose, ref[3], rtol=1e-10, atol=0)
    finally:
        device.destroy_tables(t)
        device.destroy_world(w)
