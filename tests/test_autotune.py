"""The autotuner's trials run the kernel that the run will: a palette world that
the run would give codes has them before the first trial, so that the settings
of code worlds are searched too. FP64 searches the fields that steer its
kernel, and keeps those the caller has set."""
import numpy as np
import pytest

from dxmclib_amd import backend, capi

pytestmark = pytest.mark.gpu

NAMES = ["Air, Dry (near sea level)", "Water, Liquid", "Bone, Cortical (ICRU)", "Lung (ICRU)"]
DENSITIES = [0.001205, 1.0, 1.92, 0.26]


@pytest.mark.parametrize("precision", [capi.PRECISION_FP32, capi.PRECISION_FP64])
def test_trials_run_the_kernel_of_the_run(device, precision):
    shape = (32, 40, 48)
    mat = np.zeros(shape, np.uint8)
    mat[:] = (np.arange(40) // 10)[None, :, None]
    spacing = (4.0, 4.0, 4.0)
    w = device.upload_world(mat, np.array(DENSITIES)[mat], spacing, backend.world_extent(shape[::-1], spacing), 4)
    tables = backend.HostTables(NAMES, device.world_max_density(w, 4), 90.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=90.0, al_mm=2.5, sdd=1000.0, field_size=(150.0, 110.0), histories_per_exposure=1 << 20,
                               total_exposures=4)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    tally = device.tally(mat.size)
    before = device.world_bytes(w)
    try:
        few = (capi.Exposure * 4)(*exposures)
        for x in few:
            x.n_histories = 1000
        print(f"autotune precision {precision}: a small run", flush=True)
        _, small = device.autotune(w, t, few, precision, trial_histories=1 << 16)
        assert device.world_bytes(w) == before
        print(f"autotune precision {precision}: a large run", flush=True)
        best, first = device.autotune(w, t, exposures, precision, trial_histories=1 << 16)
        assert device.world_bytes(w) >= before + mat.size
        assert first.trials > small.trials
        stats = device.run(w, t, exposures, tally, precision, seed=2, tuning=best)
        events = device.download(tally, mat.size)[1]
        device.reset_tally(tally)
        _, second = device.autotune(w, t, exposures, precision, trial_histories=1 << 16)
        assert second.trials == first.trials
        assert device.run(w, t, exposures, tally, precision, seed=2).events == stats.events
        assert np.array_equal(device.download(tally, mat.size)[1], events)
        # fields the caller sets are not searched
        for field, value in (("regeneration_threshold", 16), ("interaction_threshold", 40), ("queue_depth", 512), ("block_bounds", 1)):
            base = capi.RunCfg()
            setattr(base, field, value)
            chosen, report = device.autotune(w, t, exposures, precision, trial_histories=1 << 16, base=base)
            assert getattr(chosen, field) == value and report.trials < first.trials, field
    finally:
        device.destroy_tally(tally)
        device.destroy_tables(t)
        device.destroy_world(w)
