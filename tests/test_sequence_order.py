"""The grid and the rules of launches in sequence, compiled for the host (tests/native/sequence_order.cpp)."""

from __future__ import annotations

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_sequence_grid_covers_every_tile_once(tmp_path):
    binary = tmp_path / "sequence_order"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", str(ROOT / "stochastic-rounding-pytorch_amd" / "csrc"),
                    str(ROOT / "tests" / "native" / "sequence_order.cpp"), "-o", str(binary)], check=True)
    result = subprocess.run([str(binary)], capture_output=True, text=True, timeout=60)
    assert result.returncode == 0, result.stdout + result.stderr
    assert result.stdout.strip().endswith(", 0 failures"), result.stdout
