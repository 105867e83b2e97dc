"""sf_attn_chunk's own source on the CPU simulator against float64 attention: one range
written directly and several merged, block and causal limits, short last blocks."""

import pytest
import torch

from specfold_amd.kv_cache import PagedKVCache
from tests.simlib import build_sim_library, compiler, use_sim_library
from tests.test_gpu_append_blocks import HD, chunk_attention

pytestmark = []


@pytest.fixture(scope="module")
def sim(tmp_path_factory):
    if compiler() is None:
        pytest.skip("no clang++ (the simulator needs clang's vector extensions)")
    with use_sim_library(build_sim_library(tmp_path_factory.mktemp("simlib"))) as lib:
        yield lib


@pytest.mark.parametrize("n,prefix,block,H,Hkv", [
    (20, 0, 8, 4, 2), (40, 70, 16, 4, 2), (70, 150, 1, 6, 2), (130, 3, 32, 2, 1)])
def test_attn_chunk(sim, n, prefix, block, H, Hkv):
    g = torch.Generator().manual_seed(n + prefix)
    P = prefix + n
    q, k, v = (torch.randn(*s, generator=g).to(torch.bfloat16)
               for s in ((n, H, HD), (Hkv, P, HD), (Hkv, P, HD)))
    cache = PagedKVCache(1, Hkv, HD, P, device="cpu", page_order="shuffled", seed=2)
    cache.load_dense([(k[None], v[None])])
    vw = cache.view(0)
    o = torch.full((n + 1, H * HD), 7.0, dtype=torch.bfloat16)
    ws = torch.full((sim.attn_chunk_workspace_bytes(n, H),), 255, dtype=torch.uint8)
    sim.attn_chunk(q, vw.k, vw.v, vw.page_table, P, vw.page_size, vw.page_stride, vw.head_stride,
                   n, block, H, Hkv, HD, HD ** -0.5, o, ws)
    ref = chunk_attention(q, k, v, n, block)
    d = (o[:n].double().view(n, H, HD) - ref).abs()
    assert torch.all(d <= 2 ** -8 * ref.abs() + 2 ** -14 * v.abs().max().double())
    assert torch.all(o[n] == 7.0)
