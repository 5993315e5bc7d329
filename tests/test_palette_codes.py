"""A palette world's first run of 2^22 histories or more (the one that brings
such runs to a history for 16 voxels) gives it 1-byte codes and block codes, as
worlds of 8-byte records have from the start; runs that read no codes do not.
Its
histories stay those of reading every voxel's record: FP32 and FP64, few and
many densities a material, empty and odd densities, ragged grids, full and
part-used material maps."""
import numpy as np
import pytest

from dxmclib_amd import backend, capi

pytestmark = pytest.mark.gpu

NAMES = ["Air, Dry (near sea level)", "Water, Liquid", "Bone, Cortical (ICRU)", "Lung (ICRU)"]
DENSITIES = [0.001205, 1.0, 1.92, 0.26]


def _world(kind):
    rng = np.random.default_rng(15)
    shape = (35, 61, 50)
    names = NAMES * (16 if kind == "map64" else 1)
    z, y, x = np.ogrid[:shape[0], :shape[1], :shape[2]]
    mat = np.zeros(shape, np.uint8)
    mat[3:33, 6:55, 5:44] = 1
    mat[np.broadcast_to(((z - 17) / 9) ** 2 + ((y - 30) / 14) ** 2 + ((x - 20) / 9) ** 2 <= 1.0, shape)] = 2
    mat[8:26, 12:40, 30:42] = 3
    dens = np.array(DENSITIES, np.float32)[mat]
    if kind == "hounsfield":
        dens = np.round(dens + 0.015 * rng.standard_normal(shape), 3).clip(0.0).astype(np.float32)
    elif kind == "few_levels":
        dens = (dens * rng.choice([0.9, 1.0, 1.003, 1.1], shape)).astype(np.float32)
    elif kind == "empty":
        dens[mat == 0] = 0.0
        dens[10:14] = 0.0
    elif kind == "not_a_number":
        dens[20, 30, 25] = np.nan
    elif kind == "map64":
        mat = mat + 60
    return names, mat, dens


@pytest.mark.parametrize("kind", ["segmented", "hounsfield", "few_levels", "empty", "not_a_number", "map64"])
def test_codes_of_palette_worlds_change_nothing(device, kind):
    names, mat, dens = _world(kind)
    spacing = (1.0, 0.8, 1.2)
    n = mat.size
    w = device.upload_world(mat, dens, spacing, backend.world_extent(mat.shape[::-1], spacing), len(names))
    before = device.world_bytes(w)
    tables = backend.HostTables(names, device.world_max_density(w, len(names)), 90.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=90.0, al_mm=2.5, sdd=1000.0, field_size=(55.0, 55.0), histories_per_exposure=1_050_000,
                               total_exposures=4)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    try:
        for precision, models in ((capi.PRECISION_FP32, (0, 1, 2)), (capi.PRECISION_FP64, (1,))):
            for model in models:
                runs = []
                for flags, bb in ((capi.RUN_EXACT_STEPS, 0), (0, 1), (0, 2)):
                    print(f"palette codes {kind} precision {precision} L={model} flags {flags} block_bounds {bb}", flush=True)
                    cfg = capi.RunCfg()
                    cfg.flags = capi.RUN_COUNTERS | flags
                    cfg.block_bounds = bb
                    tally = device.tally(n)
                    stats = device.run(w, t, exposures, tally, precision, model, seed=8, tuning=cfg)
                    dose, events, _ = device.download(tally, n)
                    device.destroy_tally(tally)
                    runs.append((stats.steps, stats.events, events, dose))
                assert runs[0][1] > 0
                for r in runs[1:]:
                    assert r[:2] == runs[0][:2]
                    assert np.array_equal(r[2], runs[0][2])
                    assert np.allclose(r[3], runs[0][3], rtol=1e-9, atol=0, equal_nan=True)
        blocks = int(np.prod([-(-s // 8) for s in mat.shape]))
        assert device.world_bytes(w) == before + n + 256 * 16 + 2 * blocks
    finally:
        device.destroy_tables(t)
        device.destroy_world(w)


def _layers(n_materials, shape, steps=1):
    names = (NAMES * 16)[:n_materials]
    mat = np.zeros(shape, np.uint8)
    mat[:] = (np.arange(shape[1]) * n_materials // shape[1])[None, :, None]
    dens = np.array((DENSITIES * 16)[:n_materials], np.float32)[mat]
    if steps > 1:
        dens = dens * (1 + np.arange(shape[2], dtype=np.float32) % steps / np.float32(1000))
    return names, mat, dens


def _runs(device, names, mat, dens, settings):
    """world_bytes gained in each of the runs (precision, low-energy model, histories, run fields) on one world"""
    spacing = tuple(200.0 / s for s in mat.shape[::-1])
    w = device.upload_world(mat, dens, spacing, backend.world_extent(mat.shape[::-1], spacing), len(names))
    tables = backend.HostTables(names, device.world_max_density(w, len(names)), 90.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=90.0, al_mm=2.5, sdd=1000.0, field_size=(180.0, 180.0), histories_per_exposure=1, total_exposures=4)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    tally = device.tally(mat.size)
    gained = []
    try:
        for precision, model, histories, fields in settings:
            print(f"palette codes of {len(names)} materials, {mat.size} voxels: precision {precision} L={model} histories {histories} {fields}", flush=True)
            for x in exposures:
                x.n_histories = histories // 4
            cfg = capi.RunCfg()
            for k, v in fields.items():
                setattr(cfg, k, v)
            before = device.world_bytes(w)
            device.run(w, t, exposures, tally, precision, model, seed=3, tuning=cfg)
            gained.append(device.world_bytes(w) - before)
    finally:
        device.destroy_tally(tally)
        device.destroy_tables(t)
        device.destroy_world(w)
    return gained


def test_codes_come_with_the_histories_that_pay_for_them(device):
    enough = 1 << 22
    small = _layers(4, (32, 40, 48))
    exact = dict(flags=capi.RUN_EXACT_STEPS)
    for precision in (capi.PRECISION_FP32, capi.PRECISION_FP64):
        g = _runs(device, *small, [(precision, 1, enough, exact), (precision, 1, enough - 4, {}), (precision, 1, enough, {}), (precision, 1, enough, {})])
        assert g[0] == g[1] == g[3] == 0 and g[2] >= small[1].size
    # 7.2e7 voxels need 4.5e6 histories, of large runs that can use codes
    large = _layers(1, (112, 800, 800))
    g = _runs(device, *large, [(capi.PRECISION_FP32, 1, enough, exact), (capi.PRECISION_FP32, 1, enough, {}), (capi.PRECISION_FP32, 1, enough, {})])
    assert g[0] == g[1] == 0 and g[2] >= large[1].size


def test_worlds_that_are_as_fast_on_records_keep_them(device):
    enough = 1 << 22
    # 40 materials: the bounds are not in LDS
    segmented, levels = _layers(40, (32, 80, 48)), _layers(40, (32, 80, 48), 40)
    assert len(np.unique(segmented[2])) <= 256 < len(np.unique(levels[2].astype(np.float64) + 10 * levels[1]))
    g = _runs(device, *segmented, [(capi.PRECISION_FP64, 1, enough, {}), (capi.PRECISION_FP32, 1, enough, {}), (capi.PRECISION_FP32, 0, enough, {}),
                                   (capi.PRECISION_FP32, 1, enough, dict(block_bounds=1))])
    assert g[:3] == [0, 0, 0] and g[3] >= segmented[1].size
    g = _runs(device, *levels, [(capi.PRECISION_FP64, 1, enough, {}), (capi.PRECISION_FP32, 1, enough, {})])
    assert g[0] == 0 and g[1] >= levels[1].size
