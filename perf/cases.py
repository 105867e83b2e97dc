"""What the framework is measured on: the work a decoding program has it do.

Whole calls through the engine and the executors (a prompt's prefill, a later turn
on a cached prefix, the folded verify step), and the single pieces of a layer
through their own entry points (the MLP, the attention, the projections around it,
the output head, the greedy statistics).  Sizes are those of the named workloads in
``specfold_amd.configs`` (hidden sizes, heads, vocabularies, prefixes, 32-token
blocks, up to 8 branches, 4 sequences in one step); the models of the whole calls
keep their widths and are cut to a few layers.

Every case is a dict of plain values with a ``kind``:

  prefill  ``tokens`` prompt tokens through the executor's cache-updating forward
           (on a fresh cache, or continuing one that holds ``prefix`` tokens)
  verify   one folded verify step of ``branches`` blocks over ``prefix`` keys
  mlp      gate/up + down of ``rows`` recomputed rows out of ``branches`` blocks
  attn     attention of every row of ``branches`` blocks, ``rows`` of them recomputed
  proj     QKV + RoPE of the recomputed rows, then o_proj + residual + norm of all
  head     logits of ``width`` positions (from ``low``) of every block
  stats    greedy statistics of ``rows`` rows of logits
"""

import math

import numpy as np
import torch

from specfold_amd import _lib
from specfold_amd.configs import NLD_VOCAB, QWEN2_VOCAB_15B, QWEN2_VOCAB_7B
from specfold_amd.engine import FoldedVerifyEngine
from specfold_amd.generate.fastdllm_model_executor import FastDLLMModelExecutor
from specfold_amd.generate.nld_model_executor import NLDModelExecutor
from specfold_amd.generate.synthetic_model import ModelShape, build_nld, build_qwen2
from specfold_amd.kv_cache import PagedKVCache
from specfold_amd.synthetic import TREE_DIFFS, draft_tree_block

DEV = "cuda"
N = 32          # tokens of a block
HD = 128        # head dimension
EPS = 1e-6
BF = torch.bfloat16

# the widths of the named workloads: hidden, heads, kv heads, intermediate, vocabulary,
# and the model family ("fastdllm": QKV bias, shifted logits; "nld": neither, causal commits)
MODELS = {
    "1p5b": (1536, 12, 2, 8960, QWEN2_VOCAB_15B, "fastdllm"),
    "7b": (3584, 28, 4, 18944, QWEN2_VOCAB_7B, "fastdllm"),
    "8b": (4096, 32, 8, 14336, NLD_VOCAB, "nld"),
    "14b": (5120, 40, 8, 17408, NLD_VOCAB, "nld"),
}


def listed():
    return [
        # a 2048-token prompt before the first decoded token, the default workload's
        dict(name="prefill_7b_2048", kind="prefill", model="7b", layers=4, tokens=2048, prefix=0),
        # a further turn of a conversation: 1000 tokens (a ragged last block) after 4096
        # cached ones, causal as the diffusion LM's refresh of its cache is
        dict(name="prefill_8b_turn", kind="prefill", model="8b", layers=4, tokens=1000,
             prefix=4096),
        # the decode loop's forward: main block and 7 draft branches, most rows folded
        dict(name="verify_7b", kind="verify", model="7b", layers=8, branches=8, prefix=2112,
             delta=0.1),
        # the smallest MLP call: one block alone at the smallest width
        dict(name="mlp_1p5b_r32", kind="mlp", model="1p5b", branches=1, rows=32),
        # the MLP of a verify step where the drafts fold (7 changed rows beside the block)
        dict(name="mlp_7b_r39", kind="mlp", model="7b", branches=8, rows=39),
        # ... at the fold ratio reported for trained models, about 0.62
        dict(name="mlp_7b_r117", kind="mlp", model="7b", branches=8, rows=117),
        # ... where nothing folds: every row of 8 branches
        dict(name="mlp_14b_r256", kind="mlp", model="14b", branches=8, rows=256),
        # attention of a verify step after a 2048-token prompt
        dict(name="attn_7b_p2112", kind="attn", model="7b", branches=8, rows=39, prefix=2112,
             shuffled=False),
        # ... after a 16k prompt, its pages in any order
        dict(name="attn_14b_p16448", kind="attn", model="14b", branches=8, rows=39,
             prefix=16448, shuffled=True),
        # the projections of four sequences' verify steps run as one (5 branches each)
        dict(name="proj_8b_x4", kind="proj", model="8b", branches=20, rows=144),
        # logits of a whole verify step (the first one of a block's drafts)
        dict(name="head_7b_256", kind="head", model="7b", branches=8, low=0, width=32),
        # the statistics one decode iteration reads: a small block of 8 positions
        dict(name="stats_7b_8", kind="stats", model="7b", rows=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "verify", "mlp", "mlp", "mlp", "attn", "attn",
                       "proj", "proj", "head", "stats"])
    model = rng.choice(list(MODELS))
    c = dict(kind=kind, model=model)
    if kind == "prefill":
        # one block (a commit) to a long prompt, the wider models on shorter ones
        most = {"1p5b": 2048, "7b": 1536, "8b": 1536, "14b": 1024}[model]
        c.update(layers=2, tokens=_log_int(rng, 32, most),
                 prefix=rng.choice([0, _log_int(rng, 100, 8192)]))
    elif kind == "verify":
        c.update(layers=4, branches=rng.randint(2, 8), prefix=_log_int(rng, 512, 8192),
                 delta=rng.choice([0.1, 0.2]))
    elif kind in ("mlp", "proj"):
        rows = _log_int(rng, 8 if kind == "mlp" else 32, 1024)
        least = -(-rows // N)
        c.update(branches=rng.randint(least, max(least, min(32, 4 * least))), rows=rows)
    elif kind == "attn":
        b = rng.randint(1, 8)
        c.update(branches=b, rows=rng.randint(N, min(N * b, N + 24 * b)),
                 prefix=_log_int(rng, 64, 16448), shuffled=rng.random() < 0.5)
    elif kind == "head":
        low = 8 * rng.randint(0, 3)
        c.update(branches=rng.randint(1, 20), low=low, width=rng.choice([8, 16, 32 - low]))
        c["width"] = min(c["width"], N - low)
    else:
        c.update(rows=rng.randint(8, 32))
    return c


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rnd(g, *shape, std=1.0):
    return torch.empty(*shape, dtype=BF, device=DEV).normal_(0.0, std, generator=g)


def _ws(n):
    return torch.empty(max(int(n), 256), dtype=torch.uint8, device=DEV)


def _i32(x):
    return torch.as_tensor(np.asarray(x), dtype=torch.int32).to(DEV)


def _tree(seed, branches, rows):
    """A random branch tree and `rows` recomputed flat rows (the whole main block and
    some of the others): par [B1], rec [B1, N], src [B1, N] (nearest recomputing
    ancestor), the ascending flat rows."""
    r = np.random.default_rng(seed)
    par = np.array([0] + [int(r.integers(0, b)) for b in range(1, branches)])
    rec = np.zeros((branches, N), dtype=bool)
    if rows >= N:
        rec[0] = True
        rest = r.choice((branches - 1) * N, rows - N, replace=False) if rows > N else []
    else:               # fewer rows than a block: only the MLP takes such
        rest = r.choice(branches * N, rows, replace=False) - N
    for t in rest:
        rec[t // N + 1, t % N] = True
    src = np.zeros((branches, N), dtype=np.int64)
    for b in range(branches):
        for n in range(N):
            s = b
            while s and not rec[s, n]:
                s = par[s]
            src[b, n] = s
    return par, rec, src, np.flatnonzero(rec.reshape(-1))


def _model(case, seed):
    D, H, Hkv, I, V, family = MODELS[case["model"]]
    fast = family == "fastdllm"
    shape = ModelShape(hidden=D, heads=H, kv_heads=Hkv, layers=case["layers"], intermediate=I,
                       vocab=V, rms_eps=1e-6 if fast else 1e-5, qkv_bias=fast)
    return (build_qwen2 if fast else build_nld)(shape, seed, device=DEV, dtype=BF)


def _prefix_kv(case, seed):
    """Every layer's cached keys and values, [1, Hkv, P, hd] each."""
    g = _gen(seed + 7919)
    Hkv = MODELS[case["model"]][2]
    return [(_rnd(g, 1, Hkv, case["prefix"], HD), _rnd(g, 1, Hkv, case["prefix"], HD))
            for _ in range(case["layers"])]


def _tokens(case, seed):
    V = MODELS[case["model"]][4]
    if case["kind"] == "verify":
        g = torch.Generator().manual_seed(int(seed))
        return draft_tree_block(N, V, g, diffs=TREE_DIFFS[:case["branches"]])
    r = np.random.default_rng(seed)
    return torch.from_numpy(r.integers(0, V - 1, (1, case["tokens"])))


def _tensors(case, seed):
    """The plain (unpacked) inputs of a single piece of a layer, from the seed."""
    D, H, Hkv, I, V, family = MODELS[case["model"]]
    g = _gen(seed)
    t = {}
    kind = case["kind"]
    BN = N * case.get("branches", 0)
    if kind in ("mlp", "attn", "proj"):
        t["par"], t["rec"], t["src"], t["rows"] = _tree(seed, case["branches"], case["rows"])
    if kind == "mlp":
        t["z"] = _rnd(g, case["rows"], D)
        t["wg"], t["wu"] = _rnd(g, I, D, std=0.02), _rnd(g, I, D, std=0.02)
        t["wd"] = _rnd(g, D, I, std=0.02)
    elif kind == "attn":
        t["q"] = _rnd(g, BN + 1, H * HD)
        t["kv"] = _rnd(g, BN + 1, 2 * Hkv * HD)
        t["k"], t["v"] = _rnd(g, 1, Hkv, case["prefix"], HD), _rnd(g, 1, Hkv, case["prefix"], HD)
    elif kind == "proj":
        nq = (H + 2 * Hkv) * HD
        t["xn"], t["o"], t["x"] = _rnd(g, BN, D), _rnd(g, BN, H * HD), _rnd(g, BN, D)
        t["wqkv"], t["wo"] = _rnd(g, nq, D, std=0.02), _rnd(g, D, H * HD, std=0.02)
        t["bias"] = _rnd(g, nq, std=0.02) if family == "fastdllm" else None
        t["ln"] = (1 + 0.1 * torch.randn(D, generator=g, device=DEV)).to(BF)
        ang = torch.arange(4096, device=DEV, dtype=torch.float64)[:, None] * \
            (1e6 ** (-torch.arange(0, HD, 2, device=DEV, dtype=torch.float64) / HD))[None]
        ang = torch.cat([ang, ang], dim=1)
        t["cos"], t["sin"] = ang.cos().to(BF), ang.sin().to(BF)
        t["pos"] = 2112
    elif kind == "head":
        t["x"] = _rnd(g, BN, D)
        t["w"] = _rnd(g, V, D, std=0.02)
    elif kind == "stats":
        # confident and flat positions side by side: the spread of the logits varies
        spread = torch.linspace(0.7, 4.0, case["rows"], device=DEV)[:, None]
        t["logits"] = (torch.randn(case["rows"], V, generator=g, device=DEV) * spread).to(BF)
    return t


def prepare(case, seed):
    kind = case["kind"]
    D, H, Hkv, I, V, family = MODELS[case["model"]]
    s = dict(case=dict(case), fast=family == "fastdllm")
    if kind == "prefill":
        model = _model(case, seed)
        room = case["prefix"] + case["tokens"] + N
        ex = (FastDLLMModelExecutor if s["fast"] else NLDModelExecutor)(
            model, device=DEV, max_length=max(4096, -(-room // 1024) * 1024))
        if not s["fast"]:
            ex.set_diffusion_lm(False)       # causal, as the loop commits
        s.update(ex=ex, tokens=_tokens(case, seed).to(DEV), cache=None)
        if case["prefix"]:
            s["cache"] = ex.new_cache()
            s["cache"].load_dense(_prefix_kv(case, seed))
        return s
    if kind == "verify":
        eng = FoldedVerifyEngine(_model(case, seed))
        cache = PagedKVCache(case["layers"], Hkv, HD, case["prefix"] + 512, device=DEV)
        cache.load_dense(_prefix_kv(case, seed))
        s.update(eng=eng, cache=cache, tokens=_tokens(case, seed).to(DEV))
        return s
    t = _tensors(case, seed)
    BN = N * case.get("branches", 0)
    B1, R = case.get("branches"), case.get("rows")
    if kind in ("mlp", "attn", "proj"):
        rows = np.full(BN, BN)
        rows[:R] = t["rows"]
        s.update(rows=_i32(rows), count=_i32([R]), par=_i32(t["par"]), src=_i32(t["src"].reshape(-1)))
    if kind == "mlp":
        z = torch.zeros(BN, D, dtype=BF, device=DEV)
        z[:R] = t["z"]
        s.update(z=z, wg=_lib.pack_weight(t["wg"]), wu=_lib.pack_weight(t["wu"]),
                 wd=_lib.pack_weight(t["wd"]), act=torch.zeros(BN, I, dtype=BF, device=DEV),
                 ffn=torch.zeros(BN + 1, D, dtype=BF, device=DEV),
                 ws=_ws(max(_lib.gemm_workspace_bytes(BN, D, I),
                            _lib.gate_up_workspace_bytes(BN, D, I))))
    elif kind == "attn":
        cache = PagedKVCache(1, Hkv, HD, case["prefix"] + 512, device=DEV, seed=seed,
                             page_order="shuffled" if case["shuffled"] else "sequential")
        cache.load_dense([(t["k"], t["v"])])
        s.update(q=t["q"], kv=t["kv"], view=cache.view(0), cache=cache,
                 o=torch.zeros(BN, H * HD, dtype=BF, device=DEV),
                 ws=_ws(_lib.attn_workspace_bytes(BN, H, cache.capacity)))
    elif kind == "proj":
        nq = (H + 2 * Hkv) * HD
        z32 = dict(dtype=torch.int32, device=DEV)
        s.update(xn=t["xn"], o=t["o"], x=t["x"], bias=t["bias"], ln=t["ln"], cos=t["cos"],
                 sin=t["sin"], pos=_i32([t["pos"]]), wqkv=_lib.pack_weight(t["wqkv"]),
                 wo=_lib.pack_weight(t["wo"]), rec=torch.from_numpy(
                     t["rec"].reshape(-1).astype(np.int8)).to(DEV),
                 f=torch.zeros(BN, **z32), seg=torch.zeros(BN, **z32),
                 segcnt=torch.zeros(B1, **z32), slot=torch.zeros(BN, **z32),
                 q=torch.zeros(BN + 1, H * HD, dtype=BF, device=DEV),
                 kv=torch.zeros(BN + 1, 2 * Hkv * HD, dtype=BF, device=DEV),
                 hp=torch.zeros(BN, D, dtype=BF, device=DEV),
                 zn=torch.zeros(BN, D, dtype=BF, device=DEV),
                 ws=_ws(_lib.qkv_workspace_bytes(BN, D, nq)),
                 wso=_ws(_lib.o_proj_workspace_bytes(BN, D, H * HD)))
    elif kind == "head":
        s.update(x=t["x"], w=_lib.pack_weight(t["w"]),
                 logits=torch.zeros(BN, V, dtype=BF, device=DEV))
    elif kind == "stats":
        s["logits"] = t["logits"]
    return s


# ---- one pass -------------------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    D, H, Hkv, I, V, _ = MODELS[case["model"]]
    B1 = case.get("branches", 0)
    BN = N * B1
    if kind == "prefill":
        if s["fast"]:
            out = s["ex"].forward(s["tokens"], past_key_values=s["cache"], use_cache=True,
                                  update_past_key_values=True)
        else:
            out = s["ex"].forward(s["tokens"], past_key_values=s["cache"], use_cache=True,
                                  use_causal_mask=True)
        cache = out.past_key_values
        if s["cache"] is not None:
            cache.advance(-case["tokens"])       # the turn is dropped again
        return {"logits": out.logits, "k": cache.k_pages, "v": cache.v_pages}
    if kind == "verify":
        return s["eng"].forward(s["tokens"], s["cache"], delta=case["delta"], shift=s["fast"])
    if kind == "mlp":
        _lib.ffn_gate_up(s["z"], s["count"], BN, s["wg"], s["wu"], D, I, s["act"], s["ws"])
        _lib.ffn_down_scatter(s["act"], s["count"], BN, s["rows"], s["wd"], I, D, s["ffn"], s["ws"])
        return {"act": s["act"], "ffn": s["ffn"]}
    if kind == "attn":
        v = s["view"]
        _lib.attn_rows(s["q"], s["kv"], v.k, v.v, v.page_table, v.capacity, v.page_size,
                       v.page_stride, v.head_stride, s["src"], s["rows"], s["count"], BN, B1, N,
                       0, B1, H, Hkv, HD, HD ** -0.5, None, s["o"], None, None, s["ws"],
                       prefix_len=v.length_dev)
        return s["o"]
    if kind == "proj":
        _lib.qkv_rope_gated(s["xn"], s["rec"], s["par"], B1, N, BN, s["f"], s["src"], s["rows"],
                            s["count"], s["seg"], s["segcnt"], s["slot"], s["wqkv"], s["bias"],
                            s["cos"], s["sin"], None, D, H, Hkv, HD, s["q"], s["kv"], s["ws"],
                            pos0=s["pos"])
        _lib.o_proj_post_norm(s["o"], s["x"], s["wo"], BN, H * HD, D, s["slot"], s["ln"], EPS,
                              s["hp"], s["zn"], s["wso"])
        return {"q": s["q"], "kv": s["kv"], "hp": s["hp"], "zn": s["zn"], "rows": s["rows"],
                "src": s["src"]}
    if kind == "head":
        _lib.head_logits_rows(s["x"], BN, s["w"], D, V, s["logits"], N, s["fast"], case["low"],
                              case["width"])
        return s["logits"]
    st = _lib.logit_stats(s["logits"], 0.95)
    return [st.top_idx, st.top_val, st.zfull, st.conf_full, st.znuc, st.greedy_tok, st.conf]


# ---- what a pass cannot do without ----------------------------------------------------------


def work(case):
    kind = case["kind"]
    D, H, Hkv, I, V, _ = MODELS[case["model"]]
    nq = (H + 2 * Hkv) * HD
    layer_w = nq * D + D * H * HD + 3 * D * I
    P = case.get("prefix", 0)
    if kind == "prefill":
        T, L = case["tokens"], case["layers"]
        keys = T * P + T * (T + N) / 2
        return {"bytes": 2 * (L * layer_w + V * D + T * V + T * D + L * 2 * Hkv * HD * (P + T)),
                "flops": 2 * T * (L * layer_w + V * D) + L * 4 * H * HD * keys}
    BN = N * case.get("branches", 0)
    if kind == "verify":
        # the drafts' own rows: one per tree position, beside the main block
        L, R = case["layers"], N + case["branches"] - 1
        return {"bytes": 2 * (L * layer_w + V * D + BN * V + L * 2 * Hkv * HD * P),
                "flops": 2 * L * (R * (nq * D + 3 * D * I) + BN * D * H * HD) + 2 * BN * V * D +
                L * 4 * H * HD * (R * P + BN * N)}
    R = case.get("rows", 0)
    if kind == "mlp":
        return {"bytes": 2 * (3 * D * I + R * (2 * D + I)), "flops": 6 * R * D * I}
    if kind == "attn":
        return {"bytes": 2 * (2 * Hkv * HD * (P + R) + R * H * HD + BN * H * HD),
                "flops": 4 * H * HD * (R * P + BN * N)}
    if kind == "proj":
        return {"bytes": 2 * (nq * D + R * (D + nq) + D * H * HD + BN * (H * HD + 2 * D) + R * D),
                "flops": 2 * R * nq * D + 2 * BN * D * H * HD}
    if kind == "head":
        M = case["branches"] * case["width"]
        return {"bytes": 2 * (V * D + M * D + M * V), "flops": 2 * M * V * D}
    return {"bytes": 2 * R * V, "flops": 4 * R * V}


# the distance seen between the path and 64 bits, which is bf16's rounding of each
# stage's result: 2e-3 for one product, 4e-3 through the MLP, 1-4e-2 through a model
SEEN = {"prefill": 2e-2, "verify": 2e-2, "mlp": 4e-3, "attn": 1.7e-3, "proj": 3.2e-3,
        "head": 1.7e-3, "stats": 1.8e-3}


def tolerance(case):
    """Four times what is seen; whole numbers have to be the same."""
    return {"rel": 4 * SEEN[case["kind"]], "differ": 0.0}


# ---- the same in 64 bits --------------------------------------------------------------------


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _lin(x, w, b=None, part=16384):
    """x @ w^T (+ b), the weight taken to 64 bits a part at a time."""
    y = torch.cat([x @ w[i:i + part].double().t() for i in range(0, w.shape[0], part)], dim=-1)
    return y if b is None else y + b.double()


def _rope(x, cos, sin):
    """x [..., heads, hd] with cos / sin [..., 1, hd]."""
    x1, x2 = x[..., :HD // 2], x[..., HD // 2:]
    return x * cos + torch.cat([-x2, x1], dim=-1) * sin


def _exact_model(case, seed):
    D, H, Hkv, I, V, family = MODELS[case["model"]]
    G = H // Hkv
    m = _model(case, seed)
    base, head = m.model, m.lm_head
    eps = m.config.rms_norm_eps
    P = case["prefix"]
    prefix = _prefix_kv(case, seed) if P else None
    tokens = _tokens(case, seed).to(DEV)
    B1, T = tokens.shape
    h = base.embed_tokens.weight[tokens].double()                       # [B1, T, D]
    rot = base.rotary_emb
    ang = torch.arange(P, P + T, device=DEV, dtype=torch.float64)[:, None] * \
        rot.inv_freq.double()[None]
    ang = torch.cat([ang, ang], dim=1)[None, :, None]
    cos, sin = (f(ang) * float(rot.attention_scaling) for f in (torch.cos, torch.sin))
    if case["kind"] == "prefill":
        n = torch.arange(T, device=DEV)
        last = n if family == "nld" else (n // N * N + N - 1)    # the last own key a row sees
        hidden = n[None, :] > last[:, None]
    diffs = [set(d) for d in TREE_DIFFS[:B1]]
    par = [0] + [next(j for j in range(B1) if len(diffs[j]) == len(diffs[i]) - 1 and
                      diffs[j] < diffs[i]) for i in range(1, B1)]
    cached = []
    for li, lyr in enumerate(base.layers):
        src = torch.zeros(B1, T, dtype=torch.long, device=DEV)
        for b in range(1, B1):
            p = h[par[b]]
            rec = (h[b] - p).norm(dim=-1) > case["delta"] * p.norm(dim=-1)
            src[b] = torch.where(rec, b, src[par[b]])

        def folded(x):     # every row takes its source row's
            return torch.gather(x, 0, src.view(B1, T, *[1] * (x.dim() - 2)).expand(x.shape))

        a = lyr.self_attn
        xn = _rms(h, lyr.input_layernorm.weight, eps)
        q = _rope(_lin(xn, a.q_proj.weight, a.q_proj.bias).view(B1, T, H, HD), cos, sin)
        k = _rope(_lin(xn, a.k_proj.weight, a.k_proj.bias).view(B1, T, Hkv, HD), cos, sin)
        v = _lin(xn, a.v_proj.weight, a.v_proj.bias).view(B1, T, Hkv, HD)
        q, k, v = folded(q), folded(k), folded(v)
        cached.append((k[0], v[0]))
        o = torch.empty(B1, T, H, HD, dtype=torch.float64, device=DEV)
        for b in range(B1):
            for g in range(Hkv):
                kk, vv = k[b, :, g], v[b, :, g]
                if prefix:
                    kk = torch.cat([prefix[li][0][0, g].double(), kk])
                    vv = torch.cat([prefix[li][1][0, g].double(), vv])
                sc = torch.einsum("tgd,kd->gtk", q[b, :, g * G:g * G + G], kk) * HD ** -0.5
                if case["kind"] == "prefill":
                    sc[:, :, P:].masked_fill_(hidden[None], -math.inf)
                o[b, :, g * G:g * G + G] = torch.einsum("gtk,kd->tgd", torch.softmax(sc, -1), vv)
        hp = h + _lin(o.view(B1, T, H * HD), a.o_proj.weight)
        z = _rms(hp, lyr.post_attention_layernorm.weight, eps)
        y = torch.nn.functional.silu(_lin(z, lyr.mlp.gate_proj.weight)) * \
            _lin(z, lyr.mlp.up_proj.weight)
        h = hp + folded(_lin(y, lyr.mlp.down_proj.weight))
    logits = _lin(_rms(h, base.norm.weight, eps), head.weight)
    return logits, cached, prefix


def exact(case, seed):
    kind = case["kind"]
    D, H, Hkv, I, V, family = MODELS[case["model"]]
    G = H // Hkv
    if kind == "verify":
        logits, _, _ = _exact_model(case, seed)
        if family == "fastdllm":
            logits = torch.cat([logits[:, :1], logits[:, :-1]], dim=1)
        return logits
    if kind == "prefill":
        logits, cached, prefix = _exact_model(case, seed)
        room = max(4096, -(-(case["prefix"] + case["tokens"] + N) // 1024) * 1024)
        pages = []
        for i in (0, 1):     # [layers, pages, Hkv, 16, hd], the pages in order
            p = torch.zeros(case["layers"], Hkv, room, HD, dtype=torch.float64, device=DEV)
            for li in range(case["layers"]):
                if prefix:
                    p[li, :, :case["prefix"]] = prefix[li][i][0].double()
                p[li, :, case["prefix"]:case["prefix"] + case["tokens"]] = \
                    cached[li][i].transpose(0, 1)
            pages.append(p.view(case["layers"], Hkv, room // 16, 16, HD).transpose(1, 2).contiguous())
        return {"logits": logits, "k": pages[0], "v": pages[1]}
    t = _tensors(case, seed)
    BN = N * case.get("branches", 0)
    if kind == "mlp":
        z = t["z"].double()
        y = torch.nn.functional.silu(_lin(z, t["wg"])) * _lin(z, t["wu"])
        act = torch.zeros(BN, I, dtype=torch.float64, device=DEV)
        act[:case["rows"]] = y
        ffn = torch.zeros(BN + 1, D, dtype=torch.float64, device=DEV)
        ffn[torch.from_numpy(t["rows"]).to(DEV)] = _lin(y, t["wd"])
        return {"act": act, "ffn": ffn}
    if kind == "attn":
        src = torch.from_numpy(t["src"]).to(DEV)                         # [B1, N]
        at = src * N + torch.arange(N, device=DEV)                       # source rows
        q = t["q"][:BN].double().view(BN, H, HD)[at.view(-1)]            # [BN, H, hd]
        kv = t["kv"][:BN].double().view(BN, 2 * Hkv, HD)[at.view(-1)]
        o = torch.empty(BN, H, HD, dtype=torch.float64, device=DEV)
        for b in range(case["branches"]):
            rows = slice(b * N, b * N + N)
            for g in range(Hkv):
                kk = torch.cat([t["k"][0, g].double(), kv[rows, g]])
                vv = torch.cat([t["v"][0, g].double(), kv[rows, Hkv + g]])
                sc = torch.einsum("tgd,kd->tgk", q[rows, g * G:g * G + G], kk) * HD ** -0.5
                o[rows, g * G:g * G + G] = torch.einsum("tgk,kd->tgd", torch.softmax(sc, -1), vv)
        return o.view(BN, H * HD)
    if kind == "proj":
        rec = torch.from_numpy(t["rec"].reshape(-1)).to(DEV)
        y = _lin(t["xn"].double(), t["wqkv"], t["bias"]).view(BN, H + 2 * Hkv, HD)
        pos = t["pos"] + torch.arange(BN, device=DEV) % N
        cos, sin = t["cos"][pos].double()[:, None], t["sin"][pos].double()[:, None]
        y[:, :H + Hkv] = _rope(y[:, :H + Hkv], cos, sin)
        y = torch.where(rec[:, None, None], y, 0.0)
        y = torch.cat([y, torch.zeros_like(y[:1])])
        hp = t["x"].double() + _lin(t["o"].double(), t["wo"])
        zn = torch.zeros(BN, D, dtype=torch.float64, device=DEV)
        zn[:case["rows"]] = _rms(hp, t["ln"], EPS)[rec]
        return {"q": y[:, :H].reshape(BN + 1, H * HD), "kv": y[:, H:].reshape(BN + 1, 2 * Hkv * HD),
                "hp": hp, "zn": zn, "rows": None, "src": None}
    if kind == "head":
        x = t["x"].double().view(case["branches"], N, D)
        if family == "fastdllm":
            x = torch.cat([x[:, :1], x[:, :-1]], dim=1)
        lo, hi = case["low"], case["low"] + case["width"]
        out = torch.zeros(case["branches"], N, V, dtype=torch.float64, device=DEV)
        out[:, lo:hi] = _lin(x[:, lo:hi], t["w"])
        return out.view(BN, V)
    x = t["logits"].double()
    z = (x - x.amax(-1, keepdim=True)).exp().sum(-1)
    # equal logits: the lower index first
    order = torch.sort(-x, dim=-1, stable=True)
    return [order.indices[:, :8].to(torch.int32), -order.values[:, :8], z, 1 / z, None, None, None]
