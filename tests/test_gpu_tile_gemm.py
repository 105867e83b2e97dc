"""The tile GEMM (more than 128 rows) behind the FFN and QKV entry points, at the edges
of its row blocks (64·NMT rows, blocks of at most 256), column tiles and K ranges:
against float64 products with the other GEMM tests' bound, and bit for bit against
the streaming core's results for the same rows (a row's sums do not depend on how
many rows are computed with it)."""

import pytest
import torch
import torch.nn.functional as F

from specfold_amd import _lib
from tests.test_gpu_gemm import acc_bound, close_bf16, mm64, packed, rnd, zeros_ws

pytestmark = pytest.mark.gpu


def _ffn(z, count, bucket, rows, wg, wu, wd, D, I):
    cnt = torch.tensor([count], dtype=torch.int32).cuda()
    act = torch.full((bucket, I), 3.0, dtype=torch.bfloat16, device="cuda")
    ffn = torch.full((1025, D), 3.0, dtype=torch.bfloat16, device="cuda")
    ws = zeros_ws(max(_lib.gemm_workspace_bytes(bucket, D, I),
                      _lib.gate_up_workspace_bytes(bucket, D, I)))
    _lib.ffn_gate_up(z, cnt, bucket, wg, wu, D, I, act, ws)
    _lib.ffn_down_scatter(act, cnt, bucket, rows, wd, I, D, ffn, ws)
    return act, ffn


# D = 256: 4 K stages of gate/up; I = 8320: 520 units over the spread plan (not a whole
# number of any tile width), down's K ranges of one stage; D = 896: 7 column tiles
@pytest.mark.parametrize("D,I", [(256, 8320), (896, 8960)])
@pytest.mark.parametrize("M", [129, 192, 193, 256, 257, 385, 513, 1000, 1024])
def test_ffn_rows(M, D, I):
    g = torch.Generator().manual_seed(M + D)
    z = rnd(1024, D, gen=g)
    wg, wu = rnd(I, D, std=0.05, gen=g), rnd(I, D, std=0.05, gen=g)
    wd = rnd(D, I, std=0.02, gen=g)
    pk = packed(wg), packed(wu), packed(wd)
    rows = torch.randperm(1024, generator=g).to(torch.int32).cuda()
    act, ffn = _ffn(z, M, 1024, rows, *pk, D, I)
    few, ffn_few = _ffn(z, 100, 1024, rows, *pk, D, I)
    torch.cuda.synchronize()
    r = rows.long()
    assert torch.equal(act[:100], few[:100]) and torch.equal(ffn[r[:100]], ffn_few[r[:100]])
    assert torch.all(act[M:] == 3.0) and torch.all(ffn[r[M:]] == 3.0)
    gt, up = mm64(z[:M], wg), mm64(z[:M], wu)
    ref = F.silu(gt) * up
    close_bf16(act[:M], ref, scale=ref.float().abs() * (2 + gt.float().abs()),
               atol=(acc_bound(z[:M], wg) + acc_bound(z[:M], wu)) * (1 + up.double().abs()))
    close_bf16(ffn[r[:M]], mm64(act[:M], wd), atol=acc_bound(act[:M], wd))


# T = 8 tiles of D = 128 (one K range of 2 stages), T = 16 over 24 stages in 8 ranges
@pytest.mark.parametrize("D,H,Hkv", [(128, 4, 2), (1536, 12, 2)])
@pytest.mark.parametrize("M", [129, 192, 257, 640, 1024])
def test_qkv_rows(M, D, H, Hkv):
    g = torch.Generator().manual_seed(M + D)
    nq, N = (H + 2 * Hkv) * 128, 32
    x, w = rnd(1024, D, gen=g), rnd(nq, D, std=0.05, gen=g)
    wp = packed(w)
    rows = torch.arange(1024, dtype=torch.int32).cuda()
    cos = torch.ones(N, 128, dtype=torch.bfloat16, device="cuda")   # no rotation
    sin = torch.zeros_like(cos)
    ws = zeros_ws(_lib.qkv_workspace_bytes(1024, D, nq))

    def run(count):
        q = torch.full((1025, H * 128), 3.0, dtype=torch.bfloat16, device="cuda")
        kv = torch.full((1025, 2 * Hkv * 128), 3.0, dtype=torch.bfloat16, device="cuda")
        _lib.qkv_rope(x, rows, torch.tensor([count], dtype=torch.int32).cuda(), 1024, 1024, wp,
                      None, cos, sin, None, N, D, H, Hkv, 128, q, kv, ws)
        return torch.cat([q, kv], dim=1)

    out, few = run(M), run(100)
    torch.cuda.synchronize()
    assert torch.equal(out[:100], few[:100])
    assert torch.all(out[M:] == 3.0)
    close_bf16(out[:M], mm64(x[:M], w), atol=acc_bound(x[:M], w))
