"""The pinned ring that small uploads pass through: its bookkeeping on the host
(tests/cpp/half_ring.cpp), over sizes that fill a half exactly, sizes that do
not, and mixes, and uploads that run laps ahead of a busy stream."""

import subprocess
from pathlib import Path

import numpy as np
import pytest

import vectorcore_amd as vc

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def ring(tmp_path_factory):
    exe = tmp_path_factory.mktemp("ring") / "half_ring"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", str(ROOT / "vectorcore_amd" / "csrc" / "hip"),
                    str(ROOT / "tests" / "cpp" / "half_ring.cpp"), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("sizes", [[1 << 18], [1 << 17], [1 << 16], [1 << 15], [1 << 10], [16], [1], [1200], [100_000],
                                   [(1 << 18) - 16], [1 << 18, 1 << 17], [1 << 18, 1 << 10, 4],
                                   [1 << 18, 100_000, 1200, 1], [262_144, 131_088, 65_520]])
def test_no_byte_is_reused_before_its_upload_is_read(ring, sizes):
    for seed in range(4):
        r = subprocess.run([str(ring), str(seed), *map(str, sizes)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [256, 181])  # 256 KiB, a quarter of a half, and a size that divides none
def test_uploads_ahead_of_a_busy_stream(rows):
    x = np.random.default_rng(rows).standard_normal((32, rows, 256)).astype(np.float32)
    a = vc.Tensor(np.zeros((2048, 2048), np.float32), device="hip")
    for _ in range(50):
        a = a @ a
    tensors = [vc.Tensor(v, device="hip") for v in x]
    for t, v in zip(tensors, x):
        np.testing.assert_array_equal(t.numpy(), v)
