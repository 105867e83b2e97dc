"""The head's row counts on both sides of its dispatch (passes of 128 and 256 rows, tile
GEMM): every row equals the row of a one-block call bit for bit, windowed and shifted."""

import pytest
import torch

from specfold_amd import _lib
from tests.test_gpu_gemm import packed, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [1536, 2048])
@pytest.mark.parametrize("blocks", [4, 5, 6, 7, 8, 9, 12, 13, 16, 17, 32])
def test_rows_equal_single_blocks(blocks, D):
    g = torch.Generator().manual_seed(blocks + D)
    N, V = 32, 256 * 130 + 128
    x, wp = rnd(blocks * N, D, gen=g), packed(rnd(V, D, std=0.02, gen=g))
    got = torch.full((blocks * N, V + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    _lib.head_logits(x, blocks * N, wp, D, V, got, shift_n=N)
    win = torch.full_like(got, 7.0)
    _lib.head_logits_rows(x, blocks * N, wp, D, V, win, N, False, 3, 28)
    for b in {0, blocks // 2, blocks - 1}:
        rows = slice(b * N, b * N + N)
        one = torch.empty(N, V, dtype=torch.bfloat16, device="cuda")
        _lib.head_logits(x[rows], N, wp, D, V, one)
        assert torch.equal(got[rows, :V], torch.cat([one[:1], one[:-1]]))
        assert torch.equal(win[rows, :V][3:31], one[3:31])
        assert torch.all(win[rows][:3] == 7.0) and torch.all(win[rows][31:] == 7.0)
    assert torch.all(got[:, V:] == 7.0) and torch.all(win[:, V:] == 7.0)
