"""A palette world's first run of 2^22 histories or more gives it 1-byte codes
and block codes, as worlds of 8-byte records have from the start. Its
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
