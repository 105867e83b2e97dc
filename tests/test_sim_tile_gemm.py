"""The tile GEMM's own source (csrc/sf_gemm_tile.h) on the CPU simulator: two row
blocks, and blocks of 192 and 256 rows, through the FFN and QKV entry points
(tests/sim/gemm_sim.cpp against float64 products).  A three-workgroup grid gives
gate/up its column-spread plan, the one the tile GEMM computes, at this size."""

import subprocess

import pytest

from tests.test_sim_gemm import _build


@pytest.fixture(scope="module")
def sim(tmp_path_factory):
    return _build(tmp_path_factory, ("-DSFG_GRID=3",))


@pytest.mark.parametrize("case", [
    (128, 256, 270, 288, 30, 21),   # D, I, count, bucket, M, seed: blocks of 192 rows
    (128, 384, 250, 256, 30, 22),   # one block of 256
    (128, 768, 270, 288, 30, 23),   # 12 stages of down in 3 ranges: its tiles' partial sums
    (128, 768, 250, 256, 30, 24),
], ids=lambda c: "D%d_I%d_count%d_bucket%d_M%d" % c[:5])
def test_tile_gemm(sim, case):
    r = subprocess.run([str(sim), *map(str, case)], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
