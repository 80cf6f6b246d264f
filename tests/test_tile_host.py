"""Host side of the tiled flux_div (CPU only): tests/native/tile_check.cpp
compiled for the host with hipcc."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which(HIPCC) is None:
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("tile") / "tile_check")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--offload-host-only",
                    os.path.join(HERE, "native", "tile_check.cpp"), "-o", exe], check=True, capture_output=True)

    def run(rows):
        text = "\n".join(" ".join(map(str, r)) for r in rows)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=120).stdout
        return [[float(x) for x in line.split()] for line in out.splitlines()]
    return run


def test_blocks_beyond_32_bit_offsets(check):
    """The kernel takes a block exactly where every offset within a variable
    fits its 32 bits: 1286 + 4 cells a side do, 1287 + 4 do not."""
    blocks = [(16, 16, 16, 2), (1286, 1286, 1286, 2), (1287, 1287, 1287, 2), (1288, 1288, 1288, 1),
              (4, 4, 33000000, 2), (4, 4, 34000000, 2), (46000, 46000, 1, 1)]
    got = check(blocks)
    assert [bool(fit) for fit, _ in got] == [bool(inside) for _, inside in got]
    assert [bool(fit) for fit, _ in got] == [True, True, False, True, True, False, False]
