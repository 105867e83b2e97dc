"""A prompt's blocks in one forward: sf_attn_chunk against float64 attention, and the
executors' cache-filling forward against the same blocks taken one at a time."""

import pytest
import torch

from specfold_amd import _lib
from specfold_amd.kv_cache import PagedKVCache

pytestmark = pytest.mark.gpu
HD = 128


def chunk_attention(q, k, v, n, block):
    """[n, H, hd] in float64: row m over keys [0, P - n + end of its block)."""
    H, Hkv, P = q.shape[1], k.shape[0], k.shape[1]
    m = torch.arange(n, device=q.device)
    end = P - n + ((m // block + 1) * block).clamp(max=n)
    hide = torch.arange(P, device=q.device)[None, :] >= end[:, None]
    out = torch.empty(n, H, HD, dtype=torch.float64, device=q.device)
    for h in range(H):
        s = q[:, h].double() @ k[h * Hkv // H].double().t() * HD ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(hide, float("-inf")), -1) @ v[h * Hkv // H].double()
    return out


# one query tile and many; one range per query (written directly) and several (merged);
# short last blocks; a prefix that ends inside a page, a block and a 64-key chunk
@pytest.mark.parametrize("n,prefix,block,H,Hkv,shuffled", [
    (1, 0, 1, 4, 4, False), (40, 0, 32, 4, 2, False), (64, 0, 32, 28, 4, True),
    (129, 77, 32, 12, 2, True), (40, 3001, 8, 40, 8, True), (1000, 1200, 1, 32, 8, False),
    (1024, 1024, 32, 28, 4, True), (1024, 0, 64, 40, 8, False), (200, 5000, 1, 8, 1, True)])
def test_attn_chunk(n, prefix, block, H, Hkv, shuffled):
    g = torch.Generator(device="cuda").manual_seed(n + prefix)
    P = prefix + n

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(n, H, HD), rnd(Hkv, P, HD), rnd(Hkv, P, HD)
    cache = PagedKVCache(1, Hkv, HD, P, page_order="shuffled" if shuffled else "sequential", seed=3)
    cache.load_dense([(k[None], v[None])])
    vw = cache.view(0)
    o = torch.full((n + 1, H * HD), 7.0, dtype=torch.bfloat16, device="cuda")
    ws = torch.full((_lib.attn_chunk_workspace_bytes(n, H),), 255, dtype=torch.uint8, device="cuda")
    for _ in range(2):      # twice through one workspace
        _lib.attn_chunk(q, vw.k, vw.v, vw.page_table, P, vw.page_size, vw.page_stride,
                        vw.head_stride, n, block, H, Hkv, HD, HD ** -0.5, o, ws)
    ref = chunk_attention(q, k, v, n, block)
    d = (o[:n].double().view(n, H, HD) - ref).abs()
    # bf16 rounding of the output (2^-9), and 2^-16 of the largest value for the
    # probabilities' two bf16 parts, four times over
    assert torch.all(d <= 2 ** -8 * ref.abs() + 2 ** -14 * v.abs().max().double())
    assert torch.all(o[n] == 7.0)


@pytest.mark.parametrize("n,prefix,block,H,Hkv,at", [
    (64, 0, 32, 28, 4, 40), (1000, 77, 1, 32, 8, 600), (1024, 1024, 32, 28, 4, 1500),
    (200, 5000, 16, 40, 8, 5199), (129, 0, 64, 4, 4, 128)])
def test_attn_chunk_hidden_value_not_finite(n, prefix, block, H, Hkv, at):
    """An inf among the values reaches the rows that see its position, in its dims: all
    else is as over the finite cache (the oracle: zeros in its place)."""
    g = torch.Generator(device="cuda").manual_seed(n + at)
    P = prefix + n

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(n, H, HD), rnd(Hkv, P, HD), rnd(Hkv, P, HD)
    vz = v.clone()
    v[0, at, [3, 64]], vz[0, at, [3, 64]] = float("inf"), 0
    cache = PagedKVCache(1, Hkv, HD, P, page_order="shuffled", seed=3)
    cache.load_dense([(k[None], v[None])])
    vw = cache.view(0)
    o = torch.empty(n, H * HD, dtype=torch.bfloat16, device="cuda")
    ws = torch.full((_lib.attn_chunk_workspace_bytes(n, H),), 255, dtype=torch.uint8, device="cuda")
    _lib.attn_chunk(q, vw.k, vw.v, vw.page_table, P, vw.page_size, vw.page_stride, vw.head_stride,
                    n, block, H, Hkv, HD, HD ** -0.5, o, ws)
    ref = chunk_attention(q, k, vz, n, block)
    got = o.double().view(n, H, HD)
    m = torch.arange(n, device="cuda")
    sees = at < prefix + ((m // block + 1) * block).clamp(max=n)
    hit = torch.zeros(n, H, HD, dtype=torch.bool, device="cuda")
    hit[:, :H // Hkv, [3, 64]] = sees[:, None, None]
    assert bool(sees.any()) and not torch.any(got[hit].isfinite())
    d = (got - ref).abs()
    assert torch.all((d <= 2 ** -8 * ref.abs() + 2 ** -14 * vz.abs().max().double())[~hit])


def _executor(family):
    from specfold_amd.generate.fastdllm_model_executor import FastDLLMModelExecutor
    from specfold_amd.generate.nld_model_executor import NLDModelExecutor
    from specfold_amd.generate.synthetic_model import ModelShape
    shape = ModelShape(hidden=512, heads=8, kv_heads=2, layers=3, intermediate=8320, vocab=1000,
                       qkv_bias=family == "fastdllm")
    kw = dict(block_length=32, max_length=2048, page_order="shuffled", page_seed=1)
    if family == "fastdllm":
        return FastDLLMModelExecutor.synthetic(shape, 3, **kw)
    # the q scale starts inside the prompt
    ex = NLDModelExecutor.synthetic(shape, 3, nld_kw=dict(original_max_positions=300), **kw)
    ex.set_diffusion_lm(family == "nld_diffusion")
    return ex


@pytest.mark.parametrize("family", ["fastdllm", "nld_causal", "nld_diffusion"])
@pytest.mark.parametrize("lengths", [(70,), (1150,), (32, 500, 33)])
def test_prompt_matches_blocks(family, lengths):
    """Every forward of a run of prompts (more than one run of 1024 rows; short last
    blocks; onto a filled cache) against its blocks one at a time: logits, keys and
    values within the distance two bf16 forwards of 3 layers differ by in the order of
    their sums (the same forward in blocks of 16 rows' worth of splits measures 4e-3)."""
    ex = _executor(family)
    g = torch.Generator().manual_seed(len(lengths))
    run = (lambda t, c: ex.forward(t, c, update_past_key_values=True)) if family == "fastdllm" \
        else (lambda t, c: ex.forward(t, c, use_cache=True, use_causal_mask=True))
    whole, parts = ex.new_cache(), ex.new_cache()
    for n in lengths:
        t = torch.randint(0, 900, (1, n), generator=g)
        got = run(t, whole).logits
        hidden = ex.engine.last_hidden.clone()
        ref = torch.cat([run(t[:, s:s + 32], parts).logits for s in range(0, n, 32)], dim=1)
        assert got.shape == ref.shape and got.is_contiguous()
        rel = (got.double() - ref.double()).norm() / ref.double().norm()
        assert rel < 1.6e-2, rel
        last = ex.engine.last_hidden       # the last block's
        assert hidden.shape == last.shape
        assert (hidden.double() - last.double()).norm() / last.double().norm() < 1.6e-2
    assert whole.length == parts.length == int(whole.length_dev) == sum(lengths)
    for li in range(3):
        for a, b in zip(whole[li], parts[li]):
            assert (a.double() - b.double()).norm() / b.double().norm() < 1.6e-2


def test_prompt_repeats_itself():
    """The same prompt twice, another one of other lengths in between through the same
    buffers: the same bits."""
    ex = _executor("nld_diffusion")
    g = torch.Generator().manual_seed(7)
    t, other = (torch.randint(0, 900, (1, n), generator=g) for n in (1150, 990))

    def run(t):
        cache = ex.new_cache()
        return ex.forward(t, cache, use_cache=True, use_causal_mask=True).logits.clone(), cache
    first, ca = run(t)
    run(other)
    again, cb = run(t)
    assert torch.equal(first, again)
    for li in range(3):
        for a, b in zip(ca[li], cb[li]):
            assert torch.equal(a, b)


def test_full_cache_is_refused_as_before():
    ex = _executor("fastdllm")
    cache = ex.new_cache(96)
    with pytest.raises(ValueError):
        ex.forward(torch.zeros(1, 128, dtype=torch.long), cache, update_past_key_values=True)
    assert cache.length == 96      # the blocks that fit were committed
