"""Scores of a wave are packed into its first lanes and added 16 voxels at a
time (dose, variance and event count of a voxel by adjacent lanes). Runs of 1
to 200 histories score from few and from all lanes, with remainders of 16; one
run has to add up to the same histories run one by one. Worlds whose voxel
index needs the wide form put scores into the voxels of the beam. Pencil beams
sum the scores of up to 256 voxels a block in LDS first; a run that also lists
an exposure of another beam, without histories, does not, and scores the same."""
import numpy as np
import pytest

from dxmclib_amd import backend, capi

pytestmark = pytest.mark.gpu


def _run(device, w, t, part, tally, precision, n, first):
    part[0].n_histories = n
    return device.run(w, t, part, tally, precision, 1, seed=11, first_history=first)


@pytest.mark.parametrize("precision", [capi.PRECISION_FP32, capi.PRECISION_FP64])
@pytest.mark.parametrize("measured", [False, True])
@pytest.mark.parametrize("width", [0.0, 1e-300])
def test_packed_scores_add_up(device, precision, measured, width):
    shape = (24, 20, 22)
    mat = np.zeros(shape, np.uint8)
    meas = np.zeros(shape, np.uint8)
    meas[4:20, 5:15, 5:17] = 1  # forced events score twice
    spacing = (1.0, 1.0, 1.0)
    w = device.upload_world(mat, np.ones(shape), spacing, backend.world_extent(shape[::-1], spacing), 1, meas if measured else None)
    tables = backend.HostTables(["Water, Liquid"], [1.0], 60.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_PENCIL, position=(0.3, 0.4, -30.0), direction_cosines=(1, 0, 0, 0, 1, 0), photon_energy=60.0,
                               histories_per_exposure=1, total_exposures=1)
    part = tables.exposures(spec)
    part[0].collimation_angles[1] = width
    t = device.upload_tables(tables.desc())
    try:
        for n in (1, 15, 16, 17, 33, 64, 200):
            print(f"packed scores precision {precision} measured {measured} width {width} n {n}", flush=True)
            tally = device.tally(mat.size)
            stats = _run(device, w, t, part, tally, precision, n, 100)
            whole = device.download(tally, mat.size)
            device.reset_tally(tally)
            events = sum(_run(device, w, t, part, tally, precision, 1, 100 + i).events for i in range(n))
            single = device.download(tally, mat.size)
            device.destroy_tally(tally)
            assert stats.events == events == int(whole[1].sum())
            assert np.array_equal(whole[1], single[1])
            assert np.allclose(whole[0], single[0], rtol=1e-12, atol=0)
            assert np.allclose(whole[2], single[2], rtol=1e-12, atol=0)
    finally:
        device.destroy_tables(t)
        device.destroy_world(w)


@pytest.mark.parametrize("precision", [capi.PRECISION_FP32, capi.PRECISION_FP64])
@pytest.mark.parametrize("model,histories", [(1, 60), (0, 3_001), (1, 200_000), (2, 50_000)])
def test_pencil_scores_equal_direct_scores(device, precision, model, histories):
    # a column of 700 voxels and the scatter around it: more than the cache holds
    shape = (700, 15, 17)
    mat = np.zeros(shape, np.uint8)
    spacing = (1.0, 1.0, 0.4)
    w = device.upload_world(mat, np.ones(shape), spacing, backend.world_extent(shape[::-1], spacing), 1)
    tables = backend.HostTables(["Water, Liquid"], [1.0], 80.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_PENCIL, position=(0.3, 0.4, -300.0), direction_cosines=(1, 0, 0, 0, 1, 0), photon_energy=80.0,
                               histories_per_exposure=histories, total_exposures=2)
    pencils = tables.exposures(spec)
    mixed = (capi.Exposure * 3)(pencils[0], pencils[1], pencils[0])
    mixed[2].collimation_angles[1] = 0.1
    mixed[2].n_histories = 0
    t = device.upload_tables(tables.desc())
    out = []
    try:
        for exposures in (pencils, mixed):
            print(f"pencil scores precision {precision} L={model} histories {histories} exposures {len(exposures)}", flush=True)
            tally = device.tally(mat.size)
            stats = device.run(w, t, exposures, tally, precision, model, seed=23)
            out.append((stats.events, *device.download(tally, mat.size)))
            device.destroy_tally(tally)
    finally:
        device.destroy_tables(t)
        device.destroy_world(w)
    assert out[0][0] == out[1][0] == int(out[0][2].sum())
    assert np.array_equal(out[0][2], out[1][2])
    assert np.allclose(out[0][1], out[1][1], rtol=1e-11, atol=0)
    assert np.allclose(out[0][3], out[1][3], rtol=1e-11, atol=0)


@pytest.mark.parametrize("precision", [capi.PRECISION_FP32, capi.PRECISION_FP64])
def test_wide_voxel_index(device, precision):
    # a slice of more than 2^24 voxels: no 24-bit index
    shape = (2, 4100, 4112)
    mat = np.zeros(shape, np.uint8)
    spacing = (0.1, 0.1, 5.0)
    w = device.upload_world(mat, np.ones(shape, np.float32), spacing, backend.world_extent(shape[::-1], spacing), 1)
    tables = backend.HostTables(["Water, Liquid"], [1.0], 60.0, 1.0)
    x0, y0 = 150.03, -170.02
    spec = backend.source_spec(capi.SOURCE_PENCIL, position=(x0, y0, -30.0), direction_cosines=(1, 0, 0, 0, 1, 0), photon_energy=60.0,
                               histories_per_exposure=50_000, total_exposures=1)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    tally = device.tally(mat.size)
    try:
        print(f"wide index precision {precision}", flush=True)
        stats = device.run(w, t, exposures, tally, precision, 1, seed=11)
        dose, events, _ = device.download(tally, mat.size)
    finally:
        device.destroy_tally(tally)
        device.destroy_tables(t)
        device.destroy_world(w)
    assert int(events.sum()) == stats.events > 0
    z, y, x = np.unravel_index(np.argsort(events)[-2:], shape)
    assert set(z) == {0, 1}
    assert np.all(x == int((x0 + 0.1 * 4112 / 2) / 0.1)) and np.all(y == int((y0 + 0.1 * 4100 / 2) / 0.1))
