"""The flash prefill's row arithmetic on the CPU: offsets within a key tile are
32 bit, the cache may hold more than 4 GiB (cpp/test_prefill_tile.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

from runtherder_amd import build as B

SRC = Path(__file__).resolve().parent / "cpp" / "test_prefill_tile.cpp"


@pytest.mark.skipif(shutil.which(B.HIPCC) is None and not Path(B.HIPCC).exists(),
                    reason="hipcc not available")
def test_tile_rows_match_64_bit_arithmetic(tmp_path):
    exe = tmp_path / "tile"
    res = subprocess.run([B.HIPCC, "--offload-host-only", "-O2", "-std=c++20", "-x", "hip",
                          str(SRC), "-o", str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-2000:]
