"""GPU parity: the HIP backend, called through its C ABI, against the oracle.

Bars (tolerances stated per test):
  RNG streams                      bit-exact
  LUT / majorant (FP64)            <= 1e-12 relative (the required bar is 1e-6)
  LUT / majorant (FP32)            <= 2e-6 relative to the FP64 oracle
  single interactions (FP64)       identical up to math-library rounding:
                                   >= 99 % of samples within 1e-9 relative
  source sampling + world entry    same bar as interactions
  full transport (FP64)            total energy imparted within 0.5 %, >= 99.7 %
                                   of scored voxels with |z| < 3
  full transport (FP32 vs FP64)    total energy within 0.5 %, per-voxel z test
"""
import numpy as np
import pytest

import oracle
from dxmclib_amd import backend, capi, workloads

pytestmark = pytest.mark.gpu

NAMES = ["Water, Liquid", "Bone, Cortical (ICRU)", "Lung (ICRU)", "Air, Dry (near sea level)", "Adipose Tissue (ICRP)"]
MAXD = [1.0, 1.92, 0.26, 0.001205, 0.95]


@pytest.fixture(scope="module")
def tables():
    return backend.HostTables(NAMES, MAXD, 120.0, 1.0)


@pytest.fixture(scope="module")
def orc():
    return oracle.Oracle(NAMES, MAXD, 120.0, 1.0)


@pytest.fixture(scope="module")
def dev_tables(device, tables):
    h = device.upload_tables(tables.desc())
    yield h
    device.destroy_tables(h)


@pytest.mark.parametrize("seed,first", [(42, 0), (42, 10**9), (7, 2**40 + 3)])
def test_rng_streams_bit_exact(device, seed, first):
    print(f"rng seed={seed} first={first}", flush=True)
    gpu = device.rng_streams(seed, first, 65536, 16)
    cpu = oracle.rng_streams(seed, first, 65536, 16)
    assert np.array_equal(gpu, cpu)


def test_large_transfers(device, dev_tables, orc):
    """Host transfers above 1 MiB go through two pinned chunks (of 8 MiB below
    22 MiB in all, else 16); sizes with a partial last chunk come back intact in
    both directions."""
    n = (1 << 20) + 7  # x 4 draws x 4 B = 16 MiB + 112 B
    print(f"large transfers: rng streams n={n}", flush=True)
    assert np.array_equal(device.rng_streams(42, 12345, n, 4), oracle.rng_streams(42, 12345, n, 4))
    rng = np.random.default_rng(9)
    m = 1_200_001  # energies 9.2 MiB up, attenuation 27 MiB down
    mat = rng.integers(0, len(NAMES), m)
    e = 10 ** rng.uniform(0.0, np.log10(120.0), m)
    print(f"large transfers: LUT lookups n={m}", flush=True)
    ga, gm = device.lut_lookup(dev_tables, capi.PRECISION_FP64, mat, e)
    ca, cm = orc.lut_lookup(0, mat, e)
    assert np.max(np.abs(ga - ca) / ca) <= 1e-12
    assert np.max(np.abs(gm - cm) / cm) <= 1e-12
    # into page-locked memory from dxmc_hip_host_alloc the copy is direct
    import ctypes as C
    lib = device.lib
    p = C.c_void_p()
    assert lib.dxmc_hip_host_alloc(n * 4 * 4 + 4096, C.byref(p)) == 0
    try:
        out = np.ctypeslib.as_array(C.cast(C.c_void_p(p.value + 4096), C.POINTER(C.c_uint32)), shape=(n * 4,))
        out[:] = 0
        device._check(lib.dxmc_hip_rng_streams(device.ctx, 42, 12345, n, 4, out.ctypes.data_as(C.POINTER(C.c_uint32))))
        assert np.array_equal(out.reshape(n, 4), oracle.rng_streams(42, 12345, n, 4))
    finally:
        assert lib.dxmc_hip_host_free(p) == 0
    assert lib.dxmc_hip_host_free(C.c_void_p(12345)) != 0


def _energies(n, rng):
    e = 10 ** rng.uniform(0.0, np.log10(120.0), n)
    e[:40] = np.array([1.0, 1.07, 1.0708, 1.305, 2.146, 2.4719, 2.472, 4.0381, 4.04, 30.0] * 4)  # edges and grid points
    return e


def test_lut_fp64(device, dev_tables, orc):
    rng = np.random.default_rng(1)
    n = 20000
    mat = rng.integers(0, len(NAMES), n)
    e = _energies(n, rng)
    ga, gm = device.lut_lookup(dev_tables, capi.PRECISION_FP64, mat, e)
    ca, cm = orc.lut_lookup(0, mat, e)
    assert np.max(np.abs(ga - ca) / ca) <= 1e-12
    assert np.max(np.abs(gm - cm) / cm) <= 1e-12


def test_lut_fp32(device, dev_tables, orc):
    rng = np.random.default_rng(2)
    n = 20000
    mat = rng.integers(0, len(NAMES), n)
    e = _energies(n, rng)
    ga, gm = device.lut_lookup(dev_tables, capi.PRECISION_FP32, mat, e)
    ca, cm = orc.lut_lookup(0, mat, e)
    # base-2 evaluation in FP32 (exp2/log2, re-based coefficients)
    err_a = np.abs(ga - ca) / ca
    err_m = np.abs(gm - cm) / cm
    print(f"FP32 LUT max rel error: attenuation {err_a.max():.2e}, majorant {err_m.max():.2e}")
    # Rounding the energy to float moves the evaluation point by 2^-24
    # relative; the error is that times the local log-log slope: ~3 for the
    # photoelectric segments (~2e-7) but ~1e4 inside the 1 eV edge intervals.
    # The first 40 energies sit on absorption edges on purpose: there the
    # slope of the 1 eV edge interval (~7e3) times 2^-24 bounds the error.
    assert np.percentile(err_a[40:], 99.9) <= 2e-6
    assert np.percentile(err_m[40:], 99.9) <= 2e-6
    assert err_a[40:].max() <= 1e-4
    assert err_m[40:].max() <= 1e-4
    assert err_a[:40].max() <= 2e-3
    assert err_m[:40].max() <= 2e-3


def _particles(n, energy, rng):
    p = np.zeros((n, 8))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    p[:, 3:6] = d
    p[:, 6] = energy
    p[:, 7] = rng.uniform(0.2, 1.0, n)
    return p


def _agree(a, b, rtol=1e-9):
    """fraction of rows equal within rtol (atol 1e-12 for components near zero)"""
    ok = np.all(np.abs(a - b) <= rtol * np.abs(b) + 1e-12, axis=1)
    return ok.mean()


@pytest.mark.parametrize("L", [0, 1, 2])
@pytest.mark.parametrize("kind", [0, 1, 2, 3, 4])
def test_interactions_fp64(device, dev_tables, orc, L, kind):
    print(f"interact L={L} kind={kind}", flush=True)
    rng = np.random.default_rng(10 * L + kind)
    n = 20000
    mat = rng.integers(0, len(NAMES), n)
    p = _particles(n, 10 ** rng.uniform(0.5, 2.08, n), rng)
    gp, ge, ga = device.interact(dev_tables, capi.PRECISION_FP64, L, kind, mat, p, seed=42, first=5, forced_probability=0.3)
    cp, ce, ca = orc.interact(L, kind, mat, p, seed=42, first=5, forced_probability=0.3)
    rows = np.column_stack([gp, ge]), np.column_stack([cp, ce])
    frac = _agree(*rows)
    print(f"  agreement {frac:.5f}")
    assert frac >= 0.99
    assert np.mean(ga == ca) >= 0.99
    # energy conservation of the single interaction (kinds 0-2): E_in = E_out + E_deposited
    if kind <= 2:
        assert np.allclose(gp[:, 6] + ge, p[:, 6], rtol=1e-12, atol=1e-9)


def test_sample_particles(device, dev_tables, tables):
    """DX exposure with spectrum and heel; pencil into a world."""
    wl = workloads.dx_thorax(histories_per_exposure=1000, exposures=2)
    ext = backend.world_extent(wl.material.shape[::-1], wl.spacing)
    t = backend.HostTables(wl.names, [0.001205, 1.0, 0.95, 1.92, 0.26], 120.0, 1.0)
    exps = t.exposures(wl.spec)
    spectra = [_spectrum(wl.spec)]
    orc = oracle.Oracle(wl.names, [0.001205, 1.0, 0.95, 1.92, 0.26], 120.0, 1.0)
    orc.add_source_tables(t.source_arrays(), spectra)
    w = device.upload_world(wl.material, wl.density, wl.spacing, ext, len(wl.names))
    tt = device.upload_tables(t.desc())
    try:
        gp, gi = device.sample_particles(w, tt, capi.PRECISION_FP64, exps[0], 42, 0, 50000)
        ow = oracle.world_view(wl.material, wl.density.astype(np.float64), wl.spacing, ext)
        cp, ci = orc.sample_particles(ow, exps[0], 42, 0, 50000)
        assert np.mean(gi == ci) >= 0.999
        assert _agree(gp, cp) >= 0.999
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)


def _tube_weights(kvp, al_mm):
    """A dual-source tube's alias-table input: its unnormalised spectrum
    (the oracle's literal integral) over the left-to-right sum."""
    import math
    import os
    anode = dict(np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "anode_reference.npz")))
    e = np.arange(1.0, kvp + 0.5, 1.0)
    raw = oracle.tube_spectrum(anode, kvp, math.radians(12.0), e, [(13, al_mm)], normalize=False)
    total = 0.0
    for v in raw:
        total += v
    return raw / total, e


def test_sample_particles_dual_source(device):
    """Dual-source CT: exposures of tube A (even) and tube B (odd), each with
    its own spectrum, heel and bowtie table, sampled on the device and by the
    oracle from the same tables."""
    n = 64
    mat = np.zeros((n, n, n), dtype=np.uint8)
    dens = np.ones((n, n, n), dtype=np.float32)
    spacing = (2.0, 2.0, 2.0)
    ext = backend.world_extent((n, n, n), spacing)
    ang = np.linspace(0, 0.45, 32)
    spec = backend.source_spec(capi.SOURCE_CT_AXIAL_DUAL, tube_voltage=120.0, al_mm=6.0, tube_b_voltage=80.0, tube_b_al_mm=4.0, sdd=1000.0,
                               sdd_b=900.0, fov=500.0, fov_b=330.0, collimation=40.0, exposure_angle_step_deg=5.0, histories_per_exposure=1000,
                               bowtie_angles=ang, bowtie_weights=np.exp(-6 * ang ** 2), bowtie_b_angles=ang, bowtie_b_weights=np.exp(-12 * ang ** 2),
                               mas_a=100.0, mas_b=180.0)
    t = backend.HostTables(["Water, Liquid"], [1.0], 120.0, 1.0)
    exps = t.exposures(spec)
    orc = oracle.Oracle(["Water, Liquid"], [1.0], 120.0, 1.0)
    orc.add_source_tables(t.source_arrays(), [_tube_weights(120.0, 6.0), _tube_weights(80.0, 4.0)])
    w = device.upload_world(mat, dens, spacing, ext, 1)
    tt = device.upload_tables(t.desc())
    try:
        ow = oracle.world_view(mat, dens.astype(np.float64), spacing, ext)
        for k in (0, 1, 10, 11):
            print(f"dual exposure {k}", flush=True)
            gp, gi = device.sample_particles(w, tt, capi.PRECISION_FP64, exps[k], 42, 1000 * k, 40000)
            cp, ci = orc.sample_particles(ow, exps[k], 42, 1000 * k, 40000)
            assert np.mean(gi == ci) >= 0.999
            assert _agree(gp, cp) >= 0.999
        # the tubes differ: tube B's photons are softer on average
        ea = device.sample_particles(w, tt, capi.PRECISION_FP64, exps[0], 1, 0, 40000)[0][:, 6].mean()
        eb = device.sample_particles(w, tt, capi.PRECISION_FP64, exps[1], 1, 0, 40000)[0][:, 6].mean()
        assert eb < 0.9 * ea
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)


def _spectrum(spec):
    import ctypes as C
    n = C.c_uint64()
    lib = capi.host()
    lib.dxmc_host_source_spectrum(C.byref(spec), None, None, 0, C.byref(n))
    e = np.zeros(n.value)
    w = np.zeros(n.value)
    lib.dxmc_host_source_spectrum(C.byref(spec), e.ctypes.data_as(C.POINTER(C.c_double)), w.ctypes.data_as(C.POINTER(C.c_double)), n.value,
                                  C.byref(n))
    return w, e


def _block_edge(shape):
    """Block edge of a 1-byte code world: the smallest of 8, 16, 32 and 64
    voxels whose table of 2-byte block codes fits 64 KiB."""
    for edge in (8, 16, 32, 64):
        if 2 * int(np.prod([-(-s // edge) for s in shape])) <= 65536:
            return edge
    return 64


def _block_bytes(shape):
    """Bytes of the 2-byte block codes a 1-byte code world carries: one per
    block, the last row, column and slice clipped."""
    edge = _block_edge(shape)
    return 2 * int(np.prod([-(-s // edge) for s in shape]))


def _zstats(d1, v1, d2, v2):
    m = (d1 > 0) | (d2 > 0)
    z = (d1[m] - d2[m]) / np.sqrt(np.maximum(v1[m] + v2[m], 1e-300))
    return np.mean(np.abs(z) < 3), m.sum()


def _run_device(device, wl, L, precision, tables=None, seed=42):
    ext = backend.world_extent(wl.material.shape[::-1], wl.spacing)
    maxd = [float(wl.density[wl.material == i].max()) if np.any(wl.material == i) else 0.0 for i in range(len(wl.names))]
    t = tables or backend.HostTables(wl.names, maxd, 120.0 if wl.spec.type != capi.SOURCE_PENCIL else wl.spec.photon_energy, 1.0)
    exps = t.exposures(wl.spec)
    w = device.upload_world(wl.material, wl.density, wl.spacing, ext, len(wl.names))
    tt = device.upload_tables(t.desc())
    tally = device.tally(wl.voxels)
    try:
        stats = device.run(w, tt, exps, tally, precision, L, seed=seed)
        dose, ev, var = device.download(tally, wl.voxels)
    finally:
        device.destroy_tally(tally)
        device.destroy_tables(tt)
        device.destroy_world(w)
    return dose, ev, var, stats, t, exps, ext, maxd


@pytest.mark.parametrize("L", [0, 1, 2])
def test_transport_water_pencil_fp64(device, L):
    """Config 1 in full: 64^3 water, 60 keV pencil, 1e6 histories, seed 42."""
    print(f"transport water pencil L={L}", flush=True)
    wl = workloads.water_pencil()
    dose, ev, var, stats, t, exps, ext, maxd = _run_device(device, wl, L, capi.PRECISION_FP64)
    orc = oracle.Oracle(wl.names, maxd, wl.spec.photon_energy, 1.0)
    ow = oracle.world_view(wl.material, wl.density.astype(np.float64), wl.spacing, ext)
    ref = orc.transport(ow, exps, L=L, seed=42)
    rel = abs(dose.sum() - ref["dose"].sum()) / ref["dose"].sum()
    frac, n = _zstats(dose, var, ref["dose"], ref["variance"])
    print(f"  total rel diff {rel:.2e}, |z|<3 in {frac:.5f} of {n} voxels, steps {stats.steps} vs {ref['steps']}, events {stats.events} vs {ref['events']}")
    assert rel < 5e-3
    assert frac >= 0.997
    # identical streams: step and event counts agree within 1 %
    assert abs(stats.steps - ref["steps"]) <= 0.01 * ref["steps"]
    assert abs(stats.events - ref["events"]) <= 0.01 * ref["events"]


@pytest.mark.parametrize("L", [0, 1, 2])
def test_transport_water_pencil_fp32_vs_fp64(device, L):
    print(f"water pencil fp32 vs fp64 L={L}", flush=True)
    wl = workloads.water_pencil()
    d64, _, v64, s64, *_ = _run_device(device, wl, L, capi.PRECISION_FP64)
    d32, _, v32, s32, *_ = _run_device(device, wl, L, capi.PRECISION_FP32)
    rel = abs(d32.sum() - d64.sum()) / d64.sum()
    frac, n = _zstats(d32, v32, d64, v64)
    hot = d64 > 0.1 * d64.max()
    err = np.abs(d32[hot] - d64[hot]) / d64[hot]
    print(f"FP32 vs FP64: total {rel:.2e}, |z|<3 {frac:.5f} of {n}, voxels >10% max: mean err {err.mean():.2e} max {err.max():.2e}, "
          f"steps {s32.steps} / {s64.steps}, events {s32.events} / {s64.events}")
    assert rel < 1e-5
    assert frac >= 0.997
    # identical streams: the same histories, apart from the few whose path
    # an FP32 rounding changes (1-3 of 1.45e6 steps and 1-2 of 1.27e6
    # events): a sampler that loses or repeats draws moves these by percents
    assert abs(s32.steps - s64.steps) <= 2e-5 * s64.steps
    assert abs(s32.events - s64.events) <= 2e-5 * s64.events
    # the accuracy target: below 0.1 % in voxels above 10 % of the maximum
    assert err.max() < 1e-3


@pytest.mark.parametrize("records", ["u8", "u16", "direct"])
def test_fp32_voxel_records(device, records):
    """The FP32 path stores a palette index per voxel when the world has at
    most 256 (1 byte) or 65536 (2 bytes) distinct (density, material)
    records and the 8-byte record otherwise; each layout transports like the
    FP64 path on identical streams."""
    print(f"voxel records {records}", flush=True)
    rng = np.random.default_rng(5)
    # the 8-byte case needs more than 65536 distinct records
    shape = (48, 48, 48) if records == "direct" else (40, 40, 40)
    mat = (rng.random(shape) < 0.3).astype(np.uint8)
    base = np.array([1.0, 1.92], dtype=np.float32)[mat]
    if records == "u8":
        dens = base
        distinct, vb = 2, 1
    elif records == "u16":
        levels = rng.integers(0, 500, shape)
        dens = (base * (0.98 + 0.04 * levels / 500.0)).astype(np.float32)
        distinct, vb = np.unique(np.stack([dens.ravel().view(np.uint32), mat.ravel().astype(np.uint32)]), axis=1).shape[1], 2
    else:
        dens = (base * rng.uniform(0.98, 1.02, shape)).astype(np.float32)
        assert np.unique(np.stack([dens.ravel().view(np.uint32), mat.ravel().astype(np.uint32)]), axis=1).shape[1] > 65536
        distinct, vb = 0, 8 + 1  # the record and a 1-byte bounded-density code
    # pencil through voxel centres (a beam along voxel faces lets the FP32
    # and FP64 paths pick different voxels for photons within an FP32 ulp of
    # the face, so their histories decorrelate)
    spec = backend.source_spec(capi.SOURCE_PENCIL, position=(0.5, 0.5, -2.0 * shape[0]), direction_cosines=(1, 0, 0, 0, 1, 0),
                               photon_energy=60.0, histories_per_exposure=50_000, total_exposures=4)
    wl = workloads.Workload("records", mat, dens, (1.0, 1.0, 1.0), ["Water, Liquid", "Bone, Cortical (ICRU)"], spec, 200_000)
    ext = backend.world_extent(shape[::-1], wl.spacing)
    w = device.upload_world(mat, dens, wl.spacing, ext, 2)
    try:
        n = mat.size
        assert device.world_bytes(w) == n * (1 + 8 + vb) + 8 * distinct + (16 * 256 + _block_bytes(shape) if records == "direct" else 0)
    finally:
        device.destroy_world(w)
    d64, _, v64, s64, *_ = _run_device(device, wl, 1, capi.PRECISION_FP64)
    d32, _, v32, s32, *_ = _run_device(device, wl, 1, capi.PRECISION_FP32)
    rel = abs(d32.sum() - d64.sum()) / d64.sum()
    frac, m = _zstats(d32, v32, d64, v64)
    print(f"  total rel {rel:.2e}, |z|<3 {frac:.5f} of {m}, steps {s32.steps} vs {s64.steps}, events {s32.events} vs {s64.events}")
    # identical streams: the two paths follow the same histories
    assert rel < 1e-3
    assert frac >= 0.997
    assert abs(s32.steps - s64.steps) <= 1e-3 * s64.steps
    assert abs(s32.events - s64.events) <= 1e-3 * s64.events


@pytest.mark.parametrize("n_materials,jitter,used", [(3, True, None), (70, True, None), (3, False, None), (64, True, None),
                                                     (12, True, (0, 5, 11))])
def test_bounded_steps_exact(device, n_materials, jitter, used):
    """The FP32 kernel settles most Woodcock decisions from bounds: the total
    attenuation bounded over the photon's LUT segment, and the density
    bounded by a 1-byte (up to 64 materials) or 2-byte code per voxel in
    worlds with 8-byte records (material and an interval holding the
    density), or read exactly from the palette. Only draws between the
    bounds evaluate the attenuation and read the record. The transport is
    identical to evaluating every step in full (DXMC_RUN_EXACT_STEPS). A
    1-byte code is material * bins + bin over the whole material map (64
    entries: 3 bins each; a map whose voxels use only some materials keeps
    bins for the others), and the kernel derives the material from it."""
    print(f"bounded steps, {n_materials} materials, jitter {jitter}, used {used}", flush=True)
    rng = np.random.default_rng(8)
    shape = (48, 48, 48)
    names = (NAMES * 20)[:n_materials]
    dens_of = np.array((MAXD * 20)[:n_materials], dtype=np.float32)
    dens_of[dens_of < 0.01] = 0.5  # no near-vacuum: every material interacts
    mat = rng.integers(0, n_materials, shape).astype(np.uint8) if used is None else np.array(used, np.uint8)[rng.integers(0, len(used), shape)]
    dens = (dens_of[mat] * (rng.uniform(0.9, 1.1, shape) if jitter else 1.0)).astype(np.float32)
    spacing = (1.0, 1.0, 1.0)
    ext = backend.world_extent(shape[::-1], spacing)
    w = device.upload_world(mat, dens, spacing, ext, n_materials)
    code_bytes = 1 if n_materials <= 64 else 2
    n = mat.size
    if jitter:
        assert device.world_bytes(w) == n * (1 + 8 + 8 + code_bytes) + (16 * 256 + _block_bytes(shape) if code_bytes == 1 else 16 * 65536)
    else:
        assert device.world_bytes(w) == n * (1 + 8 + 1) + 8 * n_materials
    maxd = device.world_max_density(w, n_materials)
    t = backend.HostTables(names, maxd, 120.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=120.0, al_mm=2.5, sdd=1000.0, field_size=(48.0, 48.0),
                               histories_per_exposure=20_000, total_exposures=10)
    exps = t.exposures(spec)
    tt = device.upload_tables(t.desc())
    out = []
    try:
        # bounds (the 7-wave kernel on 1-byte codes), every step in full, and
        # the 6-wave kernel
        for flags, waves in ((capi.RUN_COUNTERS, 0), (capi.RUN_COUNTERS | capi.RUN_EXACT_STEPS, 0), (capi.RUN_COUNTERS, 6)):
            cfg = capi.RunCfg()
            cfg.flags = flags
            cfg.waves_per_simd = waves
            tally = device.tally(n)
            stats = device.run(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=3, tuning=cfg)
            d, ev, v = device.download(tally, n)
            device.destroy_tally(tally)
            out.append((stats.steps, stats.events, d, ev))
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)
    print(f"  steps {[o[0] for o in out]}, events {[o[1] for o in out]}")
    assert out[0][0] > 0
    for o in out[1:]:
        assert o[0] == out[0][0] and o[1] == out[0][1]
        assert np.array_equal(o[3], out[0][3])
        # FP64 atomics add in run-dependent order: rounding only
        assert np.allclose(o[2], out[0][2], rtol=1e-10, atol=0)


@pytest.mark.parametrize("shape,edge", [((45, 50, 53), 8), ((64, 520, 530), 16)])
def test_block_bounds_exact(device, shape, edge):
    """Worlds with 1-byte codes also carry a code range per block of
    voxels (8 to 64 per edge, the smallest block whose table fits 64 KiB):
    one-material blocks settle most Woodcock decisions from the block's
    density interval, without the voxel's code. A world of air, a water
    slab with a bone ellipsoid and a lung region (blocks of one material,
    blocks on the boundaries holding several, ragged sizes that clip the
    last blocks) runs the same histories as evaluating every step in full,
    and as reading every step's code (block_bounds = 2)."""
    print(f"block bounds {shape}", flush=True)
    assert _block_edge(shape) == edge
    rng = np.random.default_rng(21)
    # z, y, x: no size a multiple of the edge; geometry scaled to the grid
    nz, ny, nx = shape
    z, y, x = np.ogrid[:nz, :ny, :nx]
    mat = np.zeros(shape, np.uint8)
    mat[nz * 8 // 45:nz * 40 // 45, ny * 5 // 50:ny * 45 // 50, :] = 1
    mat[np.broadcast_to(((z - nz * 24 / 45) / (nz * 9 / 45)) ** 2 + ((y - ny / 2) / (ny * 12 / 50)) ** 2 + ((x - nx * 20 / 53) / (nx * 10 / 53)) ** 2 <= 1.0, shape)] = 2
    mat[nz * 10 // 45:nz * 30 // 45, ny * 10 // 50:ny * 26 // 50, nx * 36 // 53:nx * 50 // 53] = 3
    dens = (np.array([0.001205, 1.0, 1.92, 0.26], np.float32)[mat] * rng.uniform(0.98, 1.02, shape)).astype(np.float32)
    spacing = (1.0, 1.0, 1.0)
    ext = backend.world_extent(shape[::-1], spacing)
    names = [workloads.AIR, workloads.WATER, workloads.BONE, workloads.LUNG]
    w = device.upload_world(mat, dens, spacing, ext, 4)
    n = mat.size
    assert device.world_bytes(w) == n * (1 + 8 + 8 + 1) + 16 * 256 + _block_bytes(shape)
    maxd = device.world_max_density(w, 4)
    t = backend.HostTables(names, maxd, 120.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=120.0, al_mm=2.5, sdd=1000.0, field_size=(1.2 * nx, 1.2 * ny),
                               histories_per_exposure=25_000, total_exposures=8)
    exps = t.exposures(spec)
    tt = device.upload_tables(t.desc())
    out = []
    try:
        for L in (1, 2):
            # default waves (7 at L = 1, 5 at L = 2), every step in full, 6
            # waves, the voxel's code only
            for flags, waves, bb in ((capi.RUN_COUNTERS, 0, 1), (capi.RUN_COUNTERS | capi.RUN_EXACT_STEPS, 0, 0), (capi.RUN_COUNTERS, 6, 1),
                                     (capi.RUN_COUNTERS, 0, 2)):
                cfg = capi.RunCfg()
                cfg.flags = flags
                cfg.waves_per_simd = waves
                cfg.block_bounds = bb
                tally = device.tally(n)
                stats = device.run(w, tt, exps, tally, capi.PRECISION_FP32, L, seed=5, tuning=cfg)
                d, ev, v = device.download(tally, n)
                device.destroy_tally(tally)
                out.append((L, stats.steps, stats.events, d, ev))
        if edge == 8:
            # the autotuner also tries block_bounds 1 and 2 on such worlds;
            # its choice runs the same histories
            best, rep = device.autotune(w, tt, exps, capi.PRECISION_FP32, 1, trial_histories=1 << 18)
            print(f"  autotune: block_bounds {best.block_bounds}, waves {best.waves_per_simd}", flush=True)
            best.flags = capi.RUN_COUNTERS
            tally = device.tally(n)
            stats = device.run(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=5, tuning=best)
            device.destroy_tally(tally)
            assert (stats.steps, stats.events) == (out[0][1], out[0][2])
            # block_bounds beyond 2 is refused
            cfg = capi.RunCfg()
            cfg.block_bounds = 3
            tally = device.tally(n)
            try:
                with pytest.raises(backend.DxmcError):
                    device.run(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=5, tuning=cfg)
            finally:
                device.destroy_tally(tally)
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)
    print(f"  steps {[o[1] for o in out]}, events {[o[2] for o in out]}")
    assert len(out) == 8
    for L in (1, 2):
        runs = [o for o in out if o[0] == L]
        assert runs[0][1] > 0 and runs[0][2] > 0
        for o in runs[1:]:
            assert o[1] == runs[0][1] and o[2] == runs[0][2]
            assert np.array_equal(o[4], runs[0][4])
            assert np.allclose(o[3], runs[0][3], rtol=1e-10, atol=0)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_live_preview_and_mip(device, axis):
    """The run loop's live dose preview (ProgressBar::computeDoseProgressImage,
    progressbar.hpp:116-235, computed here on the device): after every launch
    the maximum intensity projection of the tally so far; previews never
    decrease, the last equals the projection of the final tally, and
    dxmc_hip_tally_mip projects like numpy along every axis."""
    print(f"live preview axis {axis}", flush=True)
    rng = np.random.default_rng(12)
    shape = (40, 36, 32)  # z, y, x: distinct sizes catch a transposed image
    nz, ny, nx = shape
    mat = (rng.random(shape) < 0.3).astype(np.uint8)
    dens = np.array([1.0, 1.92], dtype=np.float32)[mat]
    spacing = (1.0, 1.0, 1.0)
    ext = backend.world_extent((nx, ny, nz), spacing)
    t = backend.HostTables(["Water, Liquid", "Bone, Cortical (ICRU)"], [1.0, 1.92], 120.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=90.0, al_mm=2.5, sdd=1000.0, field_size=(30.0, 30.0),
                               histories_per_exposure=25_000, total_exposures=8)
    exps = t.exposures(spec)
    w = device.upload_world(mat, dens, spacing, ext, 2)
    tt = device.upload_tables(t.desc())
    tally = device.tally(mat.size)
    try:
        cfg = capi.RunCfg()
        cfg.histories_per_launch = 50_000
        images = []
        stats = device.run_monitored(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=42, tuning=cfg, preview=images.append,
                                     preview_axis=axis, preview_interval=0.0)
        assert stats.launches == 4 and len(images) == 4
        d, _, _ = device.download(tally, mat.size)
        vol = d.reshape(shape)
        want = vol.max(axis=2 - axis).astype(np.float32)
        assert images[-1].shape == want.shape and np.array_equal(images[-1], want)
        for a, b in zip(images, images[1:]):
            assert np.all(b >= a)
        assert images[0].max() > 0
        for ax in (0, 1, 2):
            assert np.array_equal(device.tally_mip(tally, w, (nx, ny, nz), ax), vol.max(axis=2 - ax).astype(np.float32))
    finally:
        device.destroy_tally(tally)
        device.destroy_tables(tt)
        device.destroy_world(w)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_world_scan_on_device(device, dtype):
    """The upload's passes over the voxels run on the device: each material's
    maximum density (exact; reference attenuationinterpolator.hpp:52-58,
    0 for an unused material), the material-index check of World::validate
    (world.hpp:182-227) and whether any measurement flag is set."""
    print(f"world scan {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(11)
    shape = (37, 41, 47)  # ragged sizes; more than 65536 distinct records
    n = int(np.prod(shape))
    mat = rng.integers(0, 4, shape).astype(np.uint8)  # material 4 of 5 unused
    dens = rng.uniform(0.1, 2.5, shape).astype(dtype)
    spacing = (1.0, 1.0, 1.0)
    ext = backend.world_extent(shape[::-1], spacing)
    want = np.array([dens[mat == m].max() if (mat == m).any() else 0.0 for m in range(5)], dtype=np.float64)

    def upload(meas=None, n_materials=5):
        return device.upload_world(mat, dens, spacing, ext, n_materials, measurement=meas)

    # 8-byte records plus 1-byte bounded-density codes (256 intervals)
    w = upload()
    try:
        assert np.array_equal(device.world_max_density(w, 5), want)
        assert device.world_bytes(w) == n * (1 + 8 + 8 + 1) + 16 * 256 + _block_bytes(shape)
    finally:
        device.destroy_world(w)
    # an all-zero measurement map is dropped; one flag keeps it (and then
    # no codes: forced interactions read the record)
    meas = np.zeros(shape, np.uint8)
    w = upload(meas)
    try:
        assert device.world_bytes(w) == n * (1 + 8 + 8 + 1) + 16 * 256 + _block_bytes(shape)
    finally:
        device.destroy_world(w)
    meas[3, 4, 5] = 1
    w = upload(meas)
    try:
        assert device.world_bytes(w) == n * (1 + 8 + 8 + 1)
        assert np.array_equal(device.world_max_density(w, 5), want)
    finally:
        device.destroy_world(w)
    # index 3 is outside a 3-material map
    with pytest.raises(backend.DxmcError):
        upload(n_materials=3)
    # a uniform world: one palette record
    one = np.full(shape, 2, np.uint8)
    w = device.upload_world(one, np.full(shape, 1.5, dtype), spacing, ext, 3)
    try:
        assert device.world_bytes(w) == n * (1 + 8 + 1) + 8
        assert np.array_equal(device.world_max_density(w, 3), [0.0, 0.0, 1.5])
    finally:
        device.destroy_world(w)


def test_autotune_keeps_results(device):
    """The autotuner changes scheduling only: a run with the tuned
    configuration follows the same histories as one with the defaults."""
    wl = workloads.dx_thorax(histories_per_exposure=4000, exposures=50)
    ext = backend.world_extent(wl.material.shape[::-1], wl.spacing)
    t = backend.HostTables(wl.names, [0.001205, 1.0, 0.95, 1.92, 0.26], 120.0, 1.0)
    exps = t.exposures(wl.spec)
    w = device.upload_world(wl.material, wl.density, wl.spacing, ext, len(wl.names))
    tt = device.upload_tables(t.desc())
    try:
        best, rep = device.autotune(w, tt, exps, capi.PRECISION_FP32, 1, trial_histories=1 << 20)
        print(f"autotune: {rep.trials} trials, default {rep.default_rate:.3e} best {rep.best_rate:.3e} hist/s; "
              f"regen {best.regeneration_threshold} interact {best.interaction_threshold} queue {best.queue_depth} "
              f"blocks/CU {best.blocks_per_cu} waves/SIMD {best.waves_per_simd}", flush=True)
        assert rep.trials >= 10
        assert rep.best_rate >= rep.default_rate * 0.9
        out = []
        for cfg in (capi.RunCfg(), best):
            cfg.flags = capi.RUN_COUNTERS
            tally = device.tally(wl.voxels)
            stats = device.run(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=42, tuning=cfg)
            d, ev, v = device.download(tally, wl.voxels)
            device.destroy_tally(tally)
            out.append((stats.steps, stats.events, d, ev))
        assert out[0][0] == out[1][0] and out[0][1] == out[1][1]
        assert np.array_equal(out[0][3], out[1][3])
        # FP64 atomics add in a different order: rounding only
        assert np.allclose(out[0][2], out[1][2], rtol=1e-10, atol=0)
        # DXMC_RUN_AUTOTUNE uses the tuned values kept in the context
        cfg = capi.RunCfg()
        cfg.flags = capi.RUN_COUNTERS | capi.RUN_AUTOTUNE
        tally = device.tally(wl.voxels)
        stats = device.run(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=42, tuning=cfg)
        device.destroy_tally(tally)
        assert stats.steps == out[0][0] and stats.events == out[0][1]
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)


def _oracle_run(wl, tables, exps, maxd, ext, L, max_e, seed=42, measurement=None):
    """The oracle on the exposures and source tables the device ran."""
    orc = oracle.Oracle(wl.names, maxd, max_e, 1.0)
    spectra = [_spectrum(wl.spec)] if wl.spec.type not in (capi.SOURCE_PENCIL,) else []
    orc.add_source_tables(tables.source_arrays(), spectra)
    ow = oracle.world_view(wl.material, wl.density.astype(np.float64), wl.spacing, ext, measurement)
    return orc.transport(ow, exps, L=L, seed=seed)


@pytest.mark.parametrize("L", [1, 2])
def test_transport_dx_fp64(device, L):
    """DX projection (120 kVp spectrum, heel) through the thorax phantom at
    reduced histories: the FP64 path follows the oracle's histories."""
    print(f"transport DX L={L}", flush=True)
    wl = workloads.dx_thorax(histories_per_exposure=5000, exposures=20)
    dose, ev, var, stats, t, exps, ext, maxd = _run_device(device, wl, L, capi.PRECISION_FP64)
    ref = _oracle_run(wl, t, exps, maxd, ext, L, 120.0)
    rel = abs(dose.sum() - ref["dose"].sum()) / ref["dose"].sum()
    frac, n = _zstats(dose, var, ref["dose"], ref["variance"])
    print(f"  total rel {rel:.2e}, |z|<3 {frac:.5f} of {n}, steps {stats.steps} vs {ref['steps']}, events {stats.events} vs {ref['events']}")
    # identical streams; device and host math libraries may differ in the
    # last bit of a transcendental, which lets a rare history take another path
    assert rel < 5e-3
    assert frac >= 0.997
    assert abs(stats.steps - ref["steps"]) <= 1e-3 * ref["steps"]
    assert abs(stats.events - ref["events"]) <= 1e-3 * ref["events"]
    # the FP32 path follows the same histories
    d32, _, v32, s32, *_ = _run_device(device, wl, L, capi.PRECISION_FP32)
    rel32 = abs(d32.sum() - dose.sum()) / dose.sum()
    print(f"  FP32: total rel {rel32:.2e}, steps {s32.steps}, events {s32.events}")
    assert rel32 < 1e-3
    assert abs(s32.steps - stats.steps) <= 1e-3 * stats.steps


def test_transport_ct_spiral_fp64(device):
    """CT spiral with bowtie and heel through the 512x512x300 phantom, 36 of
    the 3600 exposures at 2000 histories: FP64 path against the oracle."""
    wl = workloads.ct_body()
    ext = backend.world_extent(wl.material.shape[::-1], wl.spacing)
    maxd = [float(wl.density[wl.material == i].max()) if np.any(wl.material == i) else 0.0 for i in range(len(wl.names))]
    t = backend.HostTables(wl.names, maxd, 120.0, 1.0)
    allx = t.exposures(wl.spec)
    sub = (capi.Exposure * 36)()
    for j in range(36):
        sub[j] = allx[j * 100]
        sub[j].n_histories = 2000
    w = device.upload_world(wl.material, wl.density, wl.spacing, ext, len(wl.names))
    tt = device.upload_tables(t.desc())
    out = {}
    try:
        for prec in (capi.PRECISION_FP64, capi.PRECISION_FP32):
            tally = device.tally(wl.voxels)
            stats = device.run(w, tt, sub, tally, prec, 1, seed=42)
            d, ev, v = device.download(tally, wl.voxels)
            device.destroy_tally(tally)
            out[prec] = (d, v, stats)
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)
    orc = oracle.Oracle(wl.names, maxd, 120.0, 1.0)
    orc.add_source_tables(t.source_arrays(), [_spectrum(wl.spec)])
    ow = oracle.world_view(wl.material, wl.density.astype(np.float64), wl.spacing, ext)
    ref = orc.transport(ow, sub, L=1, seed=42)
    d, v, s = out[capi.PRECISION_FP64]
    rel = abs(d.sum() - ref["dose"].sum()) / ref["dose"].sum()
    frac, n = _zstats(d, v, ref["dose"], ref["variance"])
    print(f"CT FP64: total rel {rel:.2e}, |z|<3 {frac:.5f} of {n}, steps {s.steps} vs {ref['steps']}, events {s.events} vs {ref['events']}",
          flush=True)
    assert rel < 5e-3
    assert frac >= 0.997
    assert abs(s.steps - ref["steps"]) <= 1e-3 * ref["steps"]
    assert abs(s.events - ref["events"]) <= 1e-3 * ref["events"]
    d32, v32, s32 = out[capi.PRECISION_FP32]
    rel32 = abs(d32.sum() - d.sum()) / d.sum()
    print(f"CT FP32: total rel {rel32:.2e}, steps {s32.steps}, events {s32.events}", flush=True)
    assert rel32 < 1e-3
    assert abs(s32.steps - s.steps) <= 1e-3 * s.steps


@pytest.fixture(scope="module")
def whole_body():
    """The whole-body configuration: 1024x1024x600 x 0.7 mm, 8 materials,
    CT axial 120 kVp, 360 exposures."""
    return workloads.whole_body()


def test_transport_whole_body_fp64(device, whole_body):
    """The 1024x1024x600 whole-body world (629M voxels; uint8 material, fp32
    density): 36 of the 360 CT-axial exposures at 2000 histories, FP64 path
    against the oracle, FP32 against FP64."""
    wl = whole_body
    print("whole body: upload and run", flush=True)
    ext = backend.world_extent(wl.material.shape[::-1], wl.spacing)
    maxd = [float(wl.density[wl.material == i].max()) if np.any(wl.material == i) else 0.0 for i in range(len(wl.names))]
    t = backend.HostTables(wl.names, maxd, 120.0, 1.0)
    allx = t.exposures(wl.spec)
    sub = (capi.Exposure * 36)()
    for j in range(36):
        sub[j] = allx[j * 10]
        sub[j].n_histories = 2000
    w = device.upload_world(wl.material, wl.density, wl.spacing, ext, len(wl.names))
    tt = device.upload_tables(t.desc())
    out = {}
    try:
        for prec in (capi.PRECISION_FP64, capi.PRECISION_FP32):
            tally = device.tally(wl.voxels)
            stats = device.run(w, tt, sub, tally, prec, 1, seed=42)
            d, ev, v = device.download(tally, wl.voxels)
            device.destroy_tally(tally)
            out[prec] = (d, v, stats)
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)
    print("whole body: oracle", flush=True)
    orc = oracle.Oracle(wl.names, maxd, 120.0, 1.0)
    orc.add_source_tables(t.source_arrays(), [_spectrum(wl.spec)])
    ow = oracle.world_view(wl.material, wl.density.astype(np.float64), wl.spacing, ext)
    ref = orc.transport(ow, sub, L=1, seed=42)
    del ow
    d, v, s = out[capi.PRECISION_FP64]
    rel = abs(d.sum() - ref["dose"].sum()) / ref["dose"].sum()
    frac, n = _zstats(d, v, ref["dose"], ref["variance"])
    print(f"whole body FP64: total rel {rel:.2e}, |z|<3 {frac:.5f} of {n}, steps {s.steps} vs {ref['steps']}, events {s.events} vs "
          f"{ref['events']}", flush=True)
    assert rel < 5e-3
    assert frac >= 0.997
    assert abs(s.steps - ref["steps"]) <= 1e-3 * ref["steps"]
    assert abs(s.events - ref["events"]) <= 1e-3 * ref["events"]
    d32, v32, s32 = out[capi.PRECISION_FP32]
    rel32 = abs(d32.sum() - d.sum()) / d.sum()
    print(f"whole body FP32: total rel {rel32:.2e}, steps {s32.steps}, events {s32.events}", flush=True)
    assert rel32 < 1e-3
    assert abs(s32.steps - s.steps) <= 1e-3 * s.steps


def _hot_voxel_stats(d32, d64, v64):
    """FP32 against FP64 on identical streams, in the voxels above 10 % of
    the maximum dose: fraction within 0.1 %, mean signed relative difference
    with its standard error, 99th percentile of |difference| / FP64 sigma."""
    hot = d64 > 0.1 * d64.max()
    rel = (d32[hot] - d64[hot]) / d64[hot]
    sig = np.sqrt(np.maximum(v64[hot], 1e-300))
    return {"voxels": int(hot.sum()), "frac": float(np.mean(np.abs(rel) < 1e-3)), "mean": float(rel.mean()),
            "se": float(rel.std() / np.sqrt(rel.size)), "hot_total": float(d32[hot].sum() / d64[hot].sum() - 1),
            "max": float(np.abs(rel).max()), "p99_sigma": float(np.percentile(np.abs(d32[hot] - d64[hot]) / sig, 99)),
            "max_sigma": float(np.max(np.abs(d32[hot] - d64[hot]) / sig))}


# (workload, exposures kept: every k-th, histories per exposure, bound on the
# fraction of hot voxels within 0.1 %; measured 0.9983, 0.9974, 0.9992)
ACCURACY = {
    "dx_thorax": (lambda: workloads.dx_thorax(histories_per_exposure=100_000, exposures=100), 1, None, 0.995),
    "ct_body": (lambda: workloads.ct_body(), 10, None, 0.995),
    "whole_body": (None, 10, 277_778, 0.995),
}


@pytest.mark.parametrize("name", list(ACCURACY))
def test_fp32_accuracy(device, name, request):
    """FP32 against FP64 per configuration on identical streams, 1e7 (DX,
    whole body) and 1e8 (CT spiral) histories: total within 1e-3; in the
    voxels above 10 % of the maximum, the stated fraction within 0.1 %, the
    differences far below the statistical uncertainty (99th percentile of
    |FP32 - FP64| under 0.01 FP64 sigma, the largest under 2 sigma), and the
    energy in those voxels within 3e-4. The differences are deposits of the
    few histories whose FP32 trajectory crosses a voxel face on the other
    side of the FP64 one: each moves a deposit to a neighbouring voxel, which
    blurs the dose very slightly, so the hot voxels lose a little (measured
    -2.8e-5 DX, -1.5e-5 CT spiral, -1.1e-4 whole body)."""
    make, stride, per, bound = ACCURACY[name]
    wl = request.getfixturevalue("whole_body") if make is None else make()
    print(f"accuracy {name}", flush=True)
    ext = backend.world_extent(wl.material.shape[::-1], wl.spacing)
    maxd = [float(wl.density[wl.material == i].max()) if np.any(wl.material == i) else 0.0 for i in range(len(wl.names))]
    t = backend.HostTables(wl.names, maxd, 120.0, 1.0)
    allx = t.exposures(wl.spec)
    idx = list(range(0, len(allx), stride))
    sub = (capi.Exposure * len(idx))()
    for j, i in enumerate(idx):
        sub[j] = allx[i]
        if per:
            sub[j].n_histories = per
    w = device.upload_world(wl.material, wl.density, wl.spacing, ext, len(wl.names))
    tt = device.upload_tables(t.desc())
    out = {}
    try:
        for prec in (capi.PRECISION_FP64, capi.PRECISION_FP32):
            tally = device.tally(wl.voxels)
            stats = device.run(w, tt, sub, tally, prec, 1, seed=42)
            d, ev, v = device.download(tally, wl.voxels)
            device.destroy_tally(tally)
            out[prec] = (d, v, stats)
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)
    d64, v64, s64 = out[capi.PRECISION_FP64]
    d32, _, s32 = out[capi.PRECISION_FP32]
    st = _hot_voxel_stats(d32, d64, v64)
    total = abs(d32.sum() - d64.sum()) / d64.sum()
    print(f"  {name}: {s64.histories} histories, total {total:.2e}, hot voxels {st}", flush=True)
    assert total < 1e-3
    assert st["frac"] >= bound
    assert abs(st["hot_total"]) < 3e-4
    assert st["p99_sigma"] < 0.01 and st["max_sigma"] < 2.0


def test_transport_forced_fp64(device):
    """Forced interactions in flagged voxels (computeInteractionsForced,
    transport.hpp:523-581): a water cylinder with a measurement region,
    isotropic-CT source; FP64 against the oracle, FP32 against FP64."""
    shape = (20, 48, 48)
    mat = np.zeros(shape, dtype=np.uint8)
    z, y, x = np.meshgrid(np.arange(20), np.arange(48), np.arange(48), indexing="ij")
    mat[(x - 23.5) ** 2 + (y - 23.5) ** 2 < 20 ** 2] = 1
    dens = np.array([0.001205, 1.0], dtype=np.float32)[mat]
    meas = np.zeros(shape, dtype=np.uint8)
    meas[6:14, 20:28, 20:28] = 1
    names = ["Air, Dry (near sea level)", "Water, Liquid"]
    # pencil along +y through the flagged block (cosines (z, x): beam = z cross x = +y)
    spec = backend.source_spec(capi.SOURCE_PENCIL, position=(0.5, -100.0, 0.5), direction_cosines=(0, 0, 1, 1, 0, 0), photon_energy=70.0,
                               histories_per_exposure=40000, total_exposures=5)
    wl = workloads.Workload("forced", mat, dens, (1.0, 1.0, 2.0), names, spec, 200000)
    ext = backend.world_extent(shape[::-1], wl.spacing)
    maxd = [0.001205, 1.0]
    t = backend.HostTables(names, maxd, 70.0, 1.0)
    exps = t.exposures(spec)
    w = device.upload_world(mat, dens, wl.spacing, ext, 2, measurement=meas)
    tt = device.upload_tables(t.desc())
    out = {}
    try:
        for prec in (capi.PRECISION_FP64, capi.PRECISION_FP32):
            tally = device.tally(mat.size)
            stats = device.run(w, tt, exps, tally, prec, 1, seed=42)
            d, ev, v = device.download(tally, mat.size)
            device.destroy_tally(tally)
            out[prec] = (d, v, stats)
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)
    orc = oracle.Oracle(names, maxd, 70.0, 1.0)
    ow = oracle.world_view(mat, dens.astype(np.float64), wl.spacing, ext, meas)
    ref = orc.transport(ow, exps, L=1, seed=42)
    d, v, s = out[capi.PRECISION_FP64]
    flagged = meas.ravel() == 1
    rel = abs(d[flagged].sum() - ref["dose"][flagged].sum()) / ref["dose"][flagged].sum()
    print(f"forced FP64: flagged rel {rel:.2e}, steps {s.steps} vs {ref['steps']}, events {s.events} vs {ref['events']}", flush=True)
    assert d[flagged].sum() > 0
    assert rel < 5e-3
    assert abs(s.steps - ref["steps"]) <= 1e-3 * ref["steps"]
    assert abs(s.events - ref["events"]) <= 1e-3 * ref["events"]
    d32, v32, s32 = out[capi.PRECISION_FP32]
    rel32 = abs(d32[flagged].sum() - d[flagged].sum()) / d[flagged].sum()
    print(f"forced FP32: flagged rel {rel32:.2e}", flush=True)
    assert rel32 < 1e-3


def test_tally_sums_and_result_arrays(device):
    """Runs accumulate into the tally's voxel sums; normalisation
    (transport.hpp:780-816) writes the result arrays from them, so repeating
    it, in either mode, starts from the same sums. A download after a run
    and before normalising returns the sums; the projection of a tally at
    rest follows its normalised dose; a further run adds to the sums."""
    print("tally sums and result arrays", flush=True)
    rng = np.random.default_rng(21)
    shape = (24, 20, 16)  # z, y, x
    mat = rng.integers(0, 3, shape).astype(np.uint8)
    dens = np.asarray(MAXD, dtype=np.float64)[mat]
    spacing = (2.0, 1.5, 1.0)
    ext = backend.world_extent(shape[::-1], spacing)
    w = device.upload_world(mat, dens, spacing, ext, len(NAMES))
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=120.0, al_mm=2.5, sdd=1000.0, field_size=(40.0, 40.0),
                               histories_per_exposure=20_000, total_exposures=5)
    t = backend.HostTables(NAMES, MAXD, 120.0, 1.0)
    exps = t.exposures(spec)
    tt = device.upload_tables(t.desc())
    n = mat.size
    tally = device.tally(n)
    try:
        stats = device.run(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=5)
        raw = device.download(tally, n)
        assert raw[1].sum() == stats.events and raw[0].sum() > 0
        again = device.download(tally, n)
        assert all(np.array_equal(a, b) for a, b in zip(raw, again))
        h = stats.histories
        device.normalize(tally, w, capi.OUTPUT_EV_PER_HISTORY, h)
        e1 = device.download(tally, n)
        device.normalize(tally, w, capi.OUTPUT_EV_PER_HISTORY, h)
        e2 = device.download(tally, n)
        assert all(np.array_equal(a, b) for a, b in zip(e1, e2))
        assert np.array_equal(e1[1], raw[1])
        d, v = oracle.normalize(raw[0], raw[2], capi.OUTPUT_EV_PER_HISTORY, h)
        assert np.allclose(e1[0], d, rtol=1e-13, atol=0)
        assert np.allclose(e1[2], v, rtol=1e-9, atol=1e-12 * np.abs(v).max())
        device.normalize(tally, w, capi.OUTPUT_DOSE, h, calibration=2.5)
        g = device.download(tally, n)
        d, v = oracle.normalize(raw[0], raw[2], capi.OUTPUT_DOSE, h, density=dens.ravel(), spacing=np.asarray(spacing), calibration=2.5)
        assert np.allclose(g[0], d, rtol=1e-13, atol=0)
        assert np.allclose(g[2], v, rtol=1e-12, atol=0)
        mip = device.tally_mip(tally, w, shape[::-1], 2)
        assert np.array_equal(mip, g[0].reshape(shape).max(axis=0).astype(np.float32))
        more = device.run(w, tt, exps, tally, capi.PRECISION_FP32, 1, seed=6)
        r2 = device.download(tally, n)
        assert r2[1].sum() == stats.events + more.events
        assert np.all(r2[1] >= raw[1])
    finally:
        device.destroy_tally(tally)
        device.destroy_tables(tt)
        device.destroy_world(w)


@pytest.mark.parametrize("L", [1, 2])
def test_fp32_variants_follow_the_same_histories(device, L):
    """Every FP32 kernel variant and scheduling field (register budget of 4 or
    6 waves per SIMD, which 5 and 7 also give, LDS staging level 1-3, blocks per
    CU, queue depth, regeneration and interaction thresholds, launch size) runs the same
    histories: equal step, event and per-voxel event counts, dose equal to
    FP64 atomic-order rounding."""
    print(f"fp32 variants, L={L}", flush=True)
    wl = workloads.dx_thorax(histories_per_exposure=3000, exposures=40)
    ext = backend.world_extent(wl.material.shape[::-1], wl.spacing)
    t = backend.HostTables(wl.names, [0.001205, 1.0, 0.95, 1.92, 0.26], 120.0, 1.0)
    exps = t.exposures(wl.spec)
    w = device.upload_world(wl.material, wl.density, wl.spacing, ext, len(wl.names))
    tt = device.upload_tables(t.desc())
    variants = [dict(), dict(waves_per_simd=4), dict(waves_per_simd=5), dict(waves_per_simd=6), dict(waves_per_simd=7), dict(lds_tables=1), dict(lds_tables=3),
                dict(blocks_per_cu=2, queue_depth=64), dict(regeneration_threshold=1, interaction_threshold=64),
                dict(waves_per_simd=6, lds_tables=3, histories_per_launch=20_000)]
    try:
        out = []
        for v in variants:
            cfg = capi.RunCfg()
            for k, val in v.items():
                setattr(cfg, k, val)
            cfg.flags = capi.RUN_COUNTERS
            tally = device.tally(wl.voxels)
            stats = device.run(w, tt, exps, tally, capi.PRECISION_FP32, L, seed=11, tuning=cfg)
            d, ev, _ = device.download(tally, wl.voxels)
            device.destroy_tally(tally)
            out.append((v, stats.steps, stats.events, d, ev))
        ref = out[0]
        for v, steps, events, d, ev in out[1:]:
            assert (steps, events) == (ref[1], ref[2]), v
            assert np.array_equal(ev, ref[4]), v
            assert np.allclose(d, ref[3], rtol=1e-10, atol=0), v
    finally:
        device.destroy_tables(tt)
        device.destroy_world(w)
