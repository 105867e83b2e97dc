"""The tile GEMM (more than 128 rows) behind the FFN and QKV entry points, at the edges
of its row blocks (64·NMT rows, blocks of at most 256), column tiles and K ranges:
against float64 products with the other GEMM tests' bound, and bit for bit against
the streaming core's results for the same rows (a row's sums do not depend on how
many rows are computed with it).  Short K ranges stay on the streaming core at some of
these row counts (make_tile_plans): both sides of that rule are among the shapes."""

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


# 144 recomputed rows of 640 (one row block) and 300 of 1024 (two), scattered; 48 column
# tiles in 5 ranges of 6 stages
@pytest.mark.parametrize("count,BN", [(144, 640), (300, 1024)])
@pytest.mark.parametrize("gated", [False, True])
def test_qkv_gathered_rows(count, BN, gated):
    """The rows of a verify step of several sequences: gathered from among more flat
    rows, through sf_qkv_rope's row list and sf_qkv_rope_gated's compaction of rec."""
    D, H, Hkv, N = 2048, 32, 8, 32
    g = torch.Generator().manual_seed(count)
    nq = (H + 2 * Hkv) * 128
    x, w = rnd(BN, D, gen=g), rnd(nq, D, std=0.05, gen=g)
    wp = packed(w)
    pick = torch.randperm(BN, generator=g)[:count].sort().values
    cos = torch.ones(N, 128, dtype=torch.bfloat16, device="cuda")   # no rotation
    sin = torch.zeros_like(cos)
    ws = zeros_ws(_lib.qkv_workspace_bytes(BN, D, nq))

    def outputs():
        return (torch.full((BN + 1, H * 128), 3.0, dtype=torch.bfloat16, device="cuda"),
                torch.full((BN + 1, 2 * Hkv * 128), 3.0, dtype=torch.bfloat16, device="cuda"))

    def run(pick):
        q, kv = outputs()
        rows = torch.full((BN,), BN, dtype=torch.int32)
        rows[:len(pick)] = pick
        _lib.qkv_rope(x, rows.cuda(), torch.tensor([len(pick)], dtype=torch.int32).cuda(), BN, BN, wp,
                      None, cos, sin, None, N, D, H, Hkv, 128, q, kv, ws)
        return torch.cat([q, kv], dim=1)

    if gated:
        q, kv = outputs()
        rec = torch.zeros(BN, dtype=torch.int8)
        rec[pick] = 1
        f, src, rows, seg, slot = (torch.zeros(BN, dtype=torch.int32, device="cuda") for _ in range(5))
        cnt = torch.zeros(1, dtype=torch.int32, device="cuda")
        segcnt = torch.zeros(BN // N, dtype=torch.int32, device="cuda")
        par = torch.arange(BN // N, dtype=torch.int32, device="cuda")   # every branch a root
        _lib.qkv_rope_gated(x, rec.cuda(), par, BN // N, N, BN, f, src, rows, cnt, seg, segcnt, slot,
                            wp, None, cos, sin, None, D, H, Hkv, 128, q, kv, ws)
        assert int(cnt) == count and torch.equal(rows[:count].cpu().long(), pick)
        out = torch.cat([q, kv], dim=1)
    else:
        out = run(pick)
    parts = [run(pick[i:i + 100]) for i in range(0, count, 100)]
    torch.cuda.synchronize()
    others = torch.ones(BN + 1, dtype=torch.bool)
    others[pick] = False
    assert torch.all(out[others] == 3.0)
    for i, few in zip(range(0, count, 100), parts):
        assert torch.equal(out[pick[i:i + 100]], few[pick[i:i + 100]])
    close_bf16(out[pick], mm64(x[pick], w), atol=acc_bound(x[pick], w))
