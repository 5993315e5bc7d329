"""Result arrays come to the host as one stream of bytes: through a 1 MiB
page-locked ring when they fit it together, else through 16 MiB chunks that
may hold the end of one array and the start of the next. Sizes at the ring's
and the chunks' ends give the arrays that downloads one by one give."""
import ctypes as C

import numpy as np
import pytest

from dxmclib_amd import backend, capi

pytestmark = pytest.mark.gpu


def _one(device, tally, n, which):
    out = [np.full(n, 7, dtype) for dtype in (np.float64, np.uint32, np.float64)]
    types = (C.c_double, C.c_uint32, C.c_double)
    args = [out[i].ctypes.data_as(C.POINTER(types[i])) if i == which else None for i in range(3)]
    device._check(device.lib.dxmc_hip_tally_download(device.ctx, tally, *args))
    for i in range(3):
        if i != which:
            assert np.all(out[i] == 7)  # arrays not asked for stay as they are
    return out[which]


@pytest.mark.parametrize("dims", [(1, 1, 1), (52428, 1, 1), (52429, 1, 1), (1 << 10, 1 << 11, 1), ((1 << 21) + 1, 1, 1), (1 << 11, 1 << 11, 1), (1999, 1709, 1)])
def test_arrays_together_and_alone(device, dims):
    print(f"result transfers {dims}", flush=True)
    shape = dims[::-1]
    n = int(np.prod(shape))
    mat = np.zeros(shape, np.uint8)
    spacing = tuple(200.0 / d for d in dims)  # a 200 mm cube of any grid
    w = device.upload_world(mat, np.ones(shape, np.float32), spacing, backend.world_extent(dims, spacing), 1)
    tables = backend.HostTables(["Water, Liquid"], [1.0], 60.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=60.0, al_mm=2.5, sdd=1000.0, field_size=(180.0, 180.0), histories_per_exposure=200_000,
                               total_exposures=2)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    tally = device.tally(n)
    try:
        stats = device.run(w, t, exposures, tally, capi.PRECISION_FP32, 1, seed=4)
        together = device.download(tally, n)
        for which in range(3):
            assert np.array_equal(together[which], _one(device, tally, n, which))
    finally:
        device.destroy_tally(tally)
        device.destroy_tables(t)
        device.destroy_world(w)
    assert int(together[1].sum()) == stats.events > 0
