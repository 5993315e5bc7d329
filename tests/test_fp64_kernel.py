"""The FP64 transport kernel settles Woodcock decisions from FP32 bounds and
takes voxel coordinates from products with the reciprocal spacing. Both must
give what the FP64 evaluation and the division give.

CPU: the coordinate rule over random and near-whole quotients, in numpy and as
the kernel's own function (nearWhole) compiled for the host.
GPU: the same histories (steps, events, event counts) with and without the
bounds, on every world layout, at ragged sizes, for each low-energy model,
with runs of one history, of fewer than a wave and of several launches.
"""
import os
import subprocess

import numpy as np
import pytest

from dxmclib_amd import backend, build, capi


def test_reciprocal_coordinate_equals_division():
    rng = np.random.default_rng(4)
    spacing = np.concatenate([rng.uniform(0.05, 7.0, 400_000), rng.choice([0.7, 0.8, 0.1, 1.0 / 3.0, 1.5, 1e-3], 400_000)])
    inv = 1.0 / spacing
    whole = rng.integers(0, 5000, spacing.size).astype(np.float64)
    # anywhere in the grid, and within a few ulp of a voxel face
    anywhere = rng.uniform(0.0, 5000.0, spacing.size) * spacing
    face = whole * spacing
    for k in range(-3, 4):
        near = face * (1.0 + k * 2.0 ** -53)
        for d in (anywhere, near):
            q = d * inv
            divide = np.abs(q - np.rint(q)) <= np.abs(q) * 2.0 ** -50
            exact = np.trunc(d / spacing)
            assert np.array_equal(np.trunc(q)[~divide], exact[~divide])
    # the rule is needed: the product alone truncates wrongly near faces
    assert np.any(np.trunc(face * inv) != np.trunc(face / spacing))


SOURCE = r"""
#include "device/persistent.hpp"
#include <cstdio>
#include <random>
int main()
{
    std::mt19937_64 rng(4);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    const double some[] = { 0.7, 0.8, 0.1, 1.0 / 3.0, 1.5, 1e-3 };
    long needed = 0;
    for (long i = 0; i < 4000000; ++i) {
        const double spacing = i % 2 ? some[rng() % 6] : 0.05 + 6.95 * u(rng), inv = 1.0 / spacing;
        const double whole = static_cast<double>(rng() % 5000);
        // anywhere in the grid, or within a few ulp of a voxel face
        const double d = i % 4 < 2 ? 5000.0 * u(rng) * spacing : whole * spacing * (1.0 + (static_cast<int>(rng() % 7) - 3) * 0x1p-53);
        const double q = d * inv, exact = d / spacing;
        const bool differ = static_cast<unsigned>(q) != static_cast<unsigned>(exact);
        needed += differ;
        if (differ && !dxmc_dev::nearWhole(q)) {
            std::printf("spacing %a, distance %a: product %a, quotient %a\n", spacing, d, q, exact);
            return 1;
        }
    }
    std::printf("%ld products truncate differently\n", needed);
    return needed > 0 ? 0 : 1;
}
"""


def test_kernel_coordinate_rule_equals_division(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "near_whole.hip", tmp_path / "near_whole"
    src.write_text(SOURCE)
    r = subprocess.run([build.HIPCC, "-O2", "-std=c++20", "-ffp-contract=off", "--offload-host-only", "-I", os.path.join(build.HERE, "csrc"), str(src),
                        "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


NAMES = ["Water, Liquid", "Bone, Cortical (ICRU)", "Lung (ICRU)", "Air, Dry (near sea level)", "Adipose Tissue (ICRP)"]
DENSITIES = [1.0, 1.92, 0.26, 0.001205, 0.95]


def _world(kind):
    rng = np.random.default_rng(12)
    shape = (41, 45, 53)
    names = (NAMES * 14)[:70 if kind == "codes16" else 5]
    dens_of = np.array((DENSITIES * 14)[:len(names)])
    z, y, x = np.ogrid[:shape[0], :shape[1], :shape[2]]
    mat = np.full(shape, 3, np.uint8)
    mat[4:37, 5:40, 3:50] = 0
    mat[np.broadcast_to(((z - 20) / 12) ** 2 + ((y - 22) / 11) ** 2 + ((x - 25) / 14) ** 2 <= 1.0, shape)] = 1
    mat[25:34, 8:20, 30:48] = 4
    if kind == "codes16":
        mat = rng.integers(0, len(names), shape).astype(np.uint8)
    dens = dens_of[mat]
    if kind in ("codes8", "codes16", "records"):
        dens = dens * rng.uniform(0.97, 1.03, shape)  # FP64 densities between FP32 values
    elif kind == "palette16":
        dens = np.round(dens * (1 + 0.02 * rng.standard_normal(shape)), 3).clip(0.0)
    meas = None
    if kind in ("records", "palette8_measured"):
        meas = np.zeros(shape, np.uint8)
        meas[10:20, 10:30, 12:24] = 1
    return names, mat, dens, meas


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["codes8", "codes16", "palette8", "palette16", "palette8_measured", "records"])
def test_filtered_decisions_equal_fp64_evaluation(device, kind):
    names, mat, dens, meas = _world(kind)
    spacing = (0.7, 0.9, 1.1)
    n = mat.size
    w = device.upload_world(mat, dens, spacing, backend.world_extent(mat.shape[::-1], spacing), len(names), meas)
    tables = backend.HostTables(names, device.world_max_density(w, len(names)), 120.0, 1.0)
    spec = backend.source_spec(capi.SOURCE_DX, tube_voltage=120.0, al_mm=2.5, sdd=1000.0, field_size=(45.0, 45.0), histories_per_exposure=7_001,
                               total_exposures=9)
    exposures = tables.exposures(spec)
    t = device.upload_tables(tables.desc())
    try:
        for model in (0, 1, 2):
            runs = []
            for flags, per_launch, first in ((capi.RUN_COUNTERS, 0, 0), (capi.RUN_COUNTERS | capi.RUN_EXACT_STEPS, 0, 0), (capi.RUN_COUNTERS, 20_011, 0)):
                print(f"fp64 {kind} L={model} flags={flags} per launch {per_launch}", flush=True)
                cfg = capi.RunCfg()
                cfg.flags = flags
                cfg.histories_per_launch = per_launch
                tally = device.tally(n)
                stats = device.run(w, t, exposures, tally, capi.PRECISION_FP64, model, seed=17, tuning=cfg)
                dose, events, variance = device.download(tally, n)
                device.destroy_tally(tally)
                runs.append((stats.steps, stats.events, events, dose, variance))
            assert runs[0][0] > 0 and runs[0][1] > 0
            for r in runs[1:]:
                assert r[:2] == runs[0][:2]
                assert np.array_equal(r[2], runs[0][2])
                # sums of FP64 atomics in another order
                assert np.allclose(r[3], runs[0][3], rtol=1e-10, atol=0)
                assert np.allclose(r[4], runs[0][4], rtol=1e-10, atol=0)
        # the smallest runs: single histories and part of a wave add up to one run
        part = (capi.Exposure * 1)()
        part[0] = exposures[0]
        sums = []
        for sizes in ((1, 1, 61), (63,)):
            tally = device.tally(n)
            first = 0
            for k in sizes:
                part[0].n_histories = k
                device.run(w, t, part, tally, capi.PRECISION_FP64, 1, seed=17, first_history=first)
                first += k
            sums.append(device.download(tally, n))
            device.destroy_tally(tally)
        assert np.array_equal(sums[0][1], sums[1][1])
        assert np.allclose(sums[0][0], sums[1][0], rtol=1e-10, atol=0)
    finally:
        device.destroy_tables(t)
        device.destroy_world(w)
