"""Result arrays come to the host as one stream of bytes: through a 1 MiB
page-locked ring when they fit it together, else through chunks (of 8 MiB
below 22 MiB in all, else of 16 MiB) that may hold the end of one array and the start of the next. Sizes at the ring's
and the chunks' ends give the arrays that downloads one by one give. Arrays in
page-locked memory go direct, each by itself: beside them pageable ones keep
the chunks, and without pageable ones a context makes no chunks (and starts no
copy threads)."""
import ctypes as C
import os

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


@pytest.mark.parametrize("dims", [(1, 1, 1), (52428, 1, 1), (52429, 1, 1), (431, 1009, 1), (1 << 10, 1 << 10, 1), (1153433, 1, 1),
                                  (1153434, 1, 1), (1 << 10, 1 << 11, 1), ((1 << 21) + 1, 1, 1), (1 << 11, 1 << 11, 1), (1999, 1709, 1)])
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


HELPERS = 7  # copy threads a context starts with its chunks


@pytest.mark.parametrize("n", [60_000, 120_000, 2_100_000])
@pytest.mark.parametrize("locked", [(1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 1, 1), (0, 0, 0)])
def test_page_locked_arrays_beside_pageable_ones(n, locked):
    print(f"result transfers of {n} voxels, page-locked {locked}", flush=True)
    shape = (1, n // 100, 100)
    spacing = (2.0, 200.0 / shape[1], 200.0)
    dtypes, types = (np.float64, np.uint32, np.float64), (C.c_double, C.c_uint32, C.c_double)
    lib = capi.hip()
    blocks = []
    with backend.Device(0) as dev:
        w = dev.upload_world(np.zeros(shape, np.uint8), np.ones(shape, np.float32), spacing, backend.world_extent(shape[::-1], spacing), 1)
        tables = backend.HostTables(["Water, Liquid"], [1.0], 60.0, 1.0)
        spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=60.0, al_mm=2.5, sdd=1000.0, field_size=(180.0, 180.0),
                                   histories_per_exposure=100_000, total_exposures=1)
        exposures = tables.exposures(spec)
        t = dev.upload_tables(tables.desc())
        tally = dev.tally(n)
        try:
            dev.run(w, t, exposures, tally, capi.PRECISION_FP32, 1, seed=4)
            with backend.Device(0) as other:  # the runtime's own threads are there by now
                other.synchronize()
            out = []
            for lock, dtype in zip(locked, dtypes):
                if lock:
                    p = C.c_void_p()
                    assert lib.dxmc_hip_host_alloc(n * np.dtype(dtype).itemsize, C.byref(p)) == 0
                    blocks.append(p)
                    out.append(np.frombuffer((C.c_char * (n * np.dtype(dtype).itemsize)).from_address(p.value), dtype))
                else:
                    out.append(np.zeros(n, dtype))
                out[-1][:] = 7
            before = len(os.listdir("/proc/self/task"))
            dev._check(lib.dxmc_hip_tally_download(dev.ctx, tally, *[a.ctypes.data_as(C.POINTER(c)) for a, c in zip(out, types)]))
            started = len(os.listdir("/proc/self/task")) - before
            want = [_one(dev, tally, n, which) for which in range(3)]
            assert want[1].sum() > 0
            for a, b in zip(out, want):
                assert np.array_equal(a, b)
            if n < 2_000_000:  # (that world's upload made the chunks)
                pageable = sum(n * np.dtype(d).itemsize for lock, d in zip(locked, dtypes) if not lock)
                assert started >= HELPERS if pageable > 1 << 20 else started < HELPERS
        finally:
            del out
            dev.destroy_tally(tally)
            dev.destroy_tables(t)
            dev.destroy_world(w)
            for p in blocks:
                assert lib.dxmc_hip_host_free(p) == 0


@pytest.mark.parametrize("n", [(1 << 20) + 3, 2_883_583, 2_883_584, 5_000_011])
def test_uploads_keep_their_order(device, n):
    """Arrays of 8, 22 and 38 MiB with ragged ends go up in two, three, two and
    three chunks: every element arrives in its place."""
    print(f"uploads of {n} energies", flush=True)
    names = ["Water, Liquid", "Bone, Cortical (ICRU)"]
    h = backend.HostTables(names, [1.0, 1.92], 120.0, 1.0)
    t = device.upload_tables(h.desc())
    rng = np.random.default_rng(3)
    mat = rng.integers(0, 2, n)
    energy = 10 ** rng.uniform(0.0, np.log10(120.0), n)
    try:
        att, maj = device.lut_lookup(t, capi.PRECISION_FP64, mat, energy)
        # the same elements by pieces that fit the ring
        for k in range(0, n, 1 << 16):
            s = slice(k, k + (1 << 16))
            a, m = device.lut_lookup(t, capi.PRECISION_FP64, mat[s], energy[s])
            assert np.array_equal(a, att[s]) and np.array_equal(m, maj[s])
    finally:
        device.destroy_tables(t)
