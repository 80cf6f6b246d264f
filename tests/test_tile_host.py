"""Host side of the tiled flux_div and rules on block shapes (CPU only): tests/native/tile_check.cpp
compiled for the host with hipcc."""
import os
import random
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

    def run(command, rows):
        text = "\n".join(" ".join(map(str, (command,) + tuple(r))) for r in rows)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=120).stdout
        got = [[float(x) for x in line.split()] for line in out.splitlines()]
        assert len(got) == len(rows)
        return got
    return run


def test_blocks_beyond_32_bit_offsets(check):
    """The kernel takes a block exactly where every offset within a variable
    fits its 32 bits: 1286 + 4 cells a side do, 1287 + 4 do not."""
    blocks = [(16, 16, 16, 2), (1286, 1286, 1286, 2), (1287, 1287, 1287, 2), (1288, 1288, 1288, 1),
              (4, 4, 33000000, 2), (4, 4, 34000000, 2), (46000, 46000, 1, 1)]
    got = check("offsets", blocks)
    assert [bool(fit) for fit, _ in got] == [bool(inside) for _, inside in got]
    assert [bool(fit) for fit, _ in got] == [True, True, False, True, True, False, False]


# halo layers and doubles per scalar record of the compositions' windows
WINDOWS = [(1, 3), (1, 5), (1, 7), (2, 3), (2, 5), (2, 7)]


def _blocks(n, most):
    rng = random.Random(11)
    side = lambda: int(round(2 ** rng.uniform(0, most)))
    return [(side(), side(), side(), 2, rng.choice((1, 2, 27, 240, 4096))) + rng.choice(WINDOWS) + (rng.randint(0, 1),)
            for _ in range(n)]


def test_plan_is_a_launchable_tiling(check):
    """Every block gets tiles that cover it, with a thread for each column, halo
    column and closing face, in workgroups and LDS that the device has, and the
    tiling is the one that a search through every count of tiles finds."""
    rows = _blocks(3000, 8) + [(n, n, 3, 2, 1, 2, 7, 1) for n in range(1, 70)]
    for (nx, ny, nz, ng, nblk, H, SS, m), (wi, wj, tx, ty, zs, nt, lds, same) in zip(rows, check("plan", rows)):
        assert 1 <= wi <= min(64, nx) and 1 <= wj <= min(64, ny)
        assert (tx - 1) * wi < nx <= tx * wi and (ty - 1) * wj < ny <= ty * wj
        assert nt in (64, 128, 192, 256) and nt >= wi * wj and nt >= 2 * H * (wi + wj) + 4
        assert 1 <= zs <= nz and -(-nz // zs) <= 64
        assert 0 < lds <= 160 * 1024
        assert same, (nx, ny, nz, nblk, H, SS, m)


@pytest.mark.parametrize("cells", [(32, 32, 32), (300, 300, 2), (512, 512, 512), (2048, 2048, 2), (2, 30000, 2),
                                   (4, 4, 1000000)])
def test_plan_costs_no_time(check, cells):
    """The plan is made on every call: a few microseconds whatever the block
    (through every count of tiles it was 226 us at 512 x 512 and 3500 at 2048 x 2048)."""
    (us, ok), = check("time", [cells + (2,)])
    print(cells, us)
    assert ok and us < 50.0


def test_stage_pushes_where_measured_faster(check):
    """The ghosts of a Butcher-table stage: pushed and exchanged times in us."""
    rows = [((24, 20, 12, 2, 240), 40, 56), ((128, 128, 128, 2, 1), 45, 58), ((4, 8, 4, 2, 12), 5.8, 7.4),
            ((4, 4, 4, 2, 512), 7.8, 10.5), ((16, 16, 16, 2, 512), 71, 90), ((40, 48, 64, 2, 2), 8.7, 12.8),
            ((2, 2, 2, 2, 27000), 185, 110), ((6, 32, 32, 2, 512), 152, 145), ((8, 8, 256, 2, 256), 232, 205),
            ((5, 6, 7, 2, 8000), 195, 168), ((2, 8, 8, 2, 216), 11.3, 9.7), ((14, 8, 8, 2, 3375), 231, 198)]
    got = [bool(p) for p, in check("pushes", [r[0] for r in rows])]
    assert got == [pushed < exchanged for _, pushed, exchanged in rows]
