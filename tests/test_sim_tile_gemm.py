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


def test_rows_beyond_4_gib(tmp_path_factory):
    """The recomputed rows of a flat table of more than 4 GiB (260 of them: the tile GEMM;
    pages never touched take no memory) give the same q, k and v as the rows alone."""
    import torch

    from tests.simlib import build_sim_library, compiler, use_sim_library
    if compiler() is None:
        pytest.skip("no clang++ (the simulator needs clang's vector extensions)")
    D, R, BN, hd = 1024, 260, (1 << 21) + 300, 128
    g = torch.Generator().manual_seed(5)
    x = torch.empty(BN, D, dtype=torch.bfloat16)
    rows = torch.cat([torch.randperm(500, generator=g)[:100].sort().values,
                      (1 << 21) + torch.randperm(300, generator=g)[:160].sort().values])
    x[rows] = torch.randn(R, D, generator=g).to(torch.bfloat16)
    w = (torch.randn(3 * hd, D, generator=g) * 0.05).to(torch.bfloat16)
    cos, sin = torch.ones(1, hd, dtype=torch.bfloat16), torch.zeros(1, hd, dtype=torch.bfloat16)
    count = torch.tensor([R], dtype=torch.int32)
    with use_sim_library(build_sim_library(tmp_path_factory.mktemp("simlib"))) as lib:
        wp = lib.pack_weight(w)

        def run(x, rows, n):
            q = torch.empty(n + 1, hd, dtype=torch.bfloat16)
            kv = torch.empty(n + 1, 2 * hd, dtype=torch.bfloat16)
            ws = torch.zeros(lib.qkv_workspace_bytes(R, D, 3 * hd), dtype=torch.uint8)
            lib.qkv_rope(x, rows.to(torch.int32), count, R, n, wp, None, cos, sin, None, 1, D, 1, 1,
                         hd, q, kv, ws)
            return torch.cat([q[rows], kv[rows]], dim=1)

        got, alone = run(x, rows, BN), run(x[rows], torch.arange(R), R)
    assert torch.equal(got, alone)
