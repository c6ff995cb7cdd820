"""bench.py without the reference engine's library (no GPU needed): the CPU baseline is null, and the
result line is still printed."""
from __future__ import annotations

import numpy as np

import bench
from oracle import refengine


def test_cpu_baseline_without_reference_engine(monkeypatch, tmp_path, capfd):
    monkeypatch.setattr(refengine, "REFQ4K", tmp_path / "libpinfer_refq4k.so")
    assert bench.cpu_baseline(tmp_path / "model.pq", ([], None), np.zeros(1, np.int32)) is None
    assert "cpu baseline skipped" in capfd.readouterr().err
