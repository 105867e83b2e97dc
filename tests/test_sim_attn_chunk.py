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


# the value's key: in the row's own 64-key chunk (own or later block), in a chunk of its own
# past the limits of a part of the tile; one range and several, causal and blocks, a prefix
@pytest.mark.parametrize("n,prefix,block,H,Hkv,at", [
    (64, 0, 32, 4, 2, 40), (64, 0, 32, 4, 2, 63), (70, 150, 1, 6, 2, 200), (130, 3, 32, 2, 1, 70),
    (150, 20, 16, 1, 1, 169), (40, 70, 16, 4, 2, 20)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_hidden_key_not_finite(sim, n, prefix, block, H, Hkv, at, bad):
    """A key (NaN) or value that is not finite reaches the rows that see its position and,
    a value, its dims only: all else is as over the finite cache (the oracle: zeros in
    its place)."""
    g = torch.Generator().manual_seed(n + prefix)
    P = prefix + n
    q, k, v = (torch.randn(*s, generator=g).to(torch.bfloat16)
               for s in ((n, H, HD), (Hkv, P, HD), (Hkv, P, HD)))
    kz, vz = k.clone(), v.clone()
    v[Hkv - 1, at, [3, 64]], vz[Hkv - 1, at, [3, 64]] = bad, 0
    if bad != bad:
        k[Hkv - 1, at, 5], kz[Hkv - 1, at, 5] = bad, 0
    cache = PagedKVCache(1, Hkv, HD, P, device="cpu", page_order="shuffled", seed=2)
    cache.load_dense([(k[None], v[None])])
    vw = cache.view(0)
    o = torch.full((n + 1, H * HD), 7.0, dtype=torch.bfloat16)
    ws = torch.full((sim.attn_chunk_workspace_bytes(n, H),), 255, dtype=torch.uint8)
    sim.attn_chunk(q, vw.k, vw.v, vw.page_table, P, vw.page_size, vw.page_stride, vw.head_stride,
                   n, block, H, Hkv, HD, HD ** -0.5, o, ws)
    ref = chunk_attention(q, kz, vz, n, block)
    m = torch.arange(n)
    sees = at < prefix + ((m // block + 1) * block).clamp(max=n)
    got = o[:n].double().view(n, H, HD)
    d = (got - ref).abs()
    ok = d <= 2 ** -8 * ref.abs() + 2 ** -14 * vz.abs().max().double()
    heads = torch.arange(H) // (H // Hkv) == Hkv - 1
    assert torch.all(ok[~sees]) and torch.all(ok[:, ~heads])
    if bad == bad:
        ok[..., [3, 64]] = True
        assert torch.all(ok)
    assert not torch.any(got[sees][:, heads][..., [3, 64]].isfinite())
    assert torch.all(o[n] == 7.0)
