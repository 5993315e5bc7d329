"""dxmc_hip_world_bytes takes no lock, so that a query does not wait for a run,
and a run on another thread adds a palette world's codes to the count: the
count has to be atomic. Checked where the type is declared, by compiling
against the library's internal header (host side only, no GPU)."""
import os
import subprocess

import pytest

from dxmclib_amd import build

SOURCE = """
#include "internal.hpp"
static_assert(std::is_same_v<decltype(dxmc_world::bytes), std::atomic<uint64_t>>);
static_assert(std::atomic<uint64_t>::is_always_lock_free);
"""


def test_world_bytes_can_be_read_while_a_run_adds_to_them(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src = tmp_path / "world_bytes.hip"
    src.write_text(SOURCE)
    r = subprocess.run([build.HIPCC, "-std=c++20", "--offload-host-only", "-fsyntax-only", "-I", os.path.join(build.ROOT, "include"),
                        "-I", os.path.join(build.HERE, "csrc"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
