"""The bench line quotes HBM counters of the kernels it ran, not of earlier ones."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402
import cgfd  # noqa: E402

TILE = dict(tx=32, ty=8, zchunk=33)


def _summary(folder, ident):
    name = "k_march_explosion800x800x400_f32_core_hbm_counters.txt"
    text = "# counters\n" + (f"sweep_id = {ident}\n" if ident else "")
    (folder / name).write_text(text + "traffic_bytes_per_launch[32x8/33] = 5.0e10\n")


@pytest.mark.parametrize("ident", [None, "0123456789ab"])
def test_counters_of_other_kernels_are_not_quoted(tmp_path, monkeypatch, ident):
    monkeypatch.setattr(bench, "PROFILES", str(tmp_path), raising=False)
    _summary(tmp_path, ident)
    assert bench.measured_traffic("explosion800x800x400", "f32", cgfd.SPLIT_CORE, TILE) == (None, None)


def test_counters_of_these_kernels_are(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "PROFILES", str(tmp_path), raising=False)
    _summary(tmp_path, bench.sweep_id())
    assert bench.measured_traffic("explosion800x800x400", "f32", cgfd.SPLIT_CORE, TILE) == (5.0e10, "32x8/33")
