"""The benchmark prints a kernel's HBM traffic only from counters of the device code that it times."""
import os
import shutil

import pytest

import conftest


@pytest.fixture()
def bench(monkeypatch):
    monkeypatch.syspath_prepend(conftest.ROOT)
    import bench
    return bench


def test_traffic_of_other_sources_is_not_printed(bench, tmp_path):
    csrc = tmp_path / "moribs-pimc_amd" / "csrc"
    shutil.copytree(os.path.join(conftest.ROOT, "moribs-pimc_amd", "csrc"), csrc)
    profiles = tmp_path / "profiles"
    profiles.mkdir()
    summary = profiles / "traffic_w.txt"
    row = "rotor[launch] 40 60002.8 7955.5 131029607\n"
    root = str(tmp_path)

    assert bench.traffic_per_launch("w", "rotor", root=root) is None  # no summary
    summary.write_text("# HBM traffic\n" + row)
    assert bench.traffic_per_launch("w", "rotor", root=root) is None  # it does not say of what
    summary.write_text(f"# HBM traffic\n# sources {bench.kernel_sources_id(root)}\n" + row)
    assert bench.traffic_per_launch("w", "rotor", root=root) == 131029607.0
    assert bench.traffic_per_launch("w", "bisect", root=root) is None

    kernels = csrc / "pimc_kernels.hpp"
    kernels.write_text("// a comment\n" + kernels.read_text().replace("\n", "\n\n", 3))
    assert bench.traffic_per_launch("w", "rotor", root=root) == 131029607.0
    kernels.write_text(kernels.read_text() + "constexpr int other = 1;\n")
    assert bench.traffic_per_launch("w", "rotor", root=root) is None


def test_old_counters_are_not_printed(bench):
    """Every committed summary either belongs to this device code or is left out of the line."""
    d = os.path.join(conftest.ROOT, "profiles")
    for tag in bench.WORKLOAD_TAG.values():
        path = os.path.join(d, f"traffic_{tag}.txt")
        if not os.path.exists(path):
            continue
        with open(path) as f:
            current = f"# sources {bench.kernel_sources_id()}" in f.read().splitlines()
        for family in ("bisect", "centroid", "rotor", "estimate"):
            assert (bench.traffic_per_launch(tag, family) is not None) == current, (tag, family)
