"""The grid columns from which a tile's padded rows are staged stay on the grid, for every
layout of the plane-tiled kernels and every axis length down to the shortest
(tests/layout/check_staging.cpp, compiled from cunfft_amd/csrc/grid_tile.hpp for the
host)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_staged_columns(tmp_path):
    exe = tmp_path / "check_staging"
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "cunfft_amd", "csrc"),
                    os.path.join(ROOT, "tests", "layout", "check_staging.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("STAGING_OK"), r.stdout
    assert "5 with spare units" in r.stdout, r.stdout
