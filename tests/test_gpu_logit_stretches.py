"""The greedy statistics at the edges of the stretches kept in LDS: rows of few, exactly
the most, one more and very many distinct 64-key stretches give the numbers of the
float64 softmax, the nucleus cut of the reference's rule (by the walk in LDS and the one
in memory) and its greedy token, and leave the histogram zero for the next call (each
row is followed by a plain one through the same workspace)."""

import pytest
import torch

from specfold_amd import _lib
from tests.test_gpu_logit_stats import nucleus_mass64

pytestmark = pytest.mark.gpu


def _row(stretches, V, seed):
    """V bf16 values over `stretches` of the finite 64-key stretches, values in [-60, 20]."""
    g = torch.Generator().manual_seed(seed)
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    vals = bits.view(torch.bfloat16)
    f = vals.float()
    ok = f.isfinite() & (f <= 20) & (f >= -60)
    group = (torch.arange(65536) // 64)
    groups = group[ok].unique()
    pick = groups[torch.randperm(len(groups), generator=g)[:stretches]]
    cand = torch.nonzero(ok & torch.isin(group, pick)).flatten()
    first = torch.stack([cand[group[cand] == p][0] for p in pick])   # each stretch once
    rest = cand[torch.randint(0, len(cand), (V - len(first),), generator=g)]
    take = torch.cat([first, rest])[torch.randperm(V, generator=g)]
    return vals[take]


@pytest.mark.parametrize("stretches", [1, 80, 159, 160, 161, 700])
def test_stretches(stretches):
    V = 16384
    x = torch.stack([_row(stretches, V, stretches),
                     torch.randn(V, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)])
    x = x.cuda()
    got = [_lib.logit_stats(x, 0.95) for _ in range(2)]     # the second on the cleared histogram
    d = x.double()
    z = (d - d.amax(-1, keepdim=True)).exp().sum(-1)
    order = torch.sort(-d, dim=-1, stable=True)
    for st in got:
        # fp32 sum of at most 16384 terms: 2^-24 * sqrt(V) * a few
        assert torch.all((st.zfull.double() - z).abs() <= 1e-4 * z)
        assert torch.equal(st.top_idx.long(), order.indices[:, :8])
        assert torch.equal(st.top_val.double(), -order.values[:, :8])
        assert torch.equal(st.znuc, got[0].znuc) and torch.equal(st.greedy_tok, got[0].greedy_tok)
    assert torch.all(got[0].znuc <= got[0].zfull * (1 + 1e-6))
    for top_p in (0.3, 0.8, 0.95, 0.999):
        st = _lib.logit_stats(x, top_p)
        zn, _ = nucleus_mass64(x, top_p)
        # the cut moves by one token (e <= 1) where the bf16 sum rounds across top_p
        assert torch.all((st.znuc.double() - zn).abs() <= 1e-4 * z + 1.0), (top_p, st.znuc, zn)
        # the kernel's own nucleus mass, fp32: its bf16 reciprocal, and the lowest index
        # whose bf16 probability is as large (torch's bf16 softmax of the kept logits is up
        # to two bf16 steps off at a flat row's mass, so it is no oracle here)
        assert torch.equal(st.conf, (1 / st.znuc).to(torch.bfloat16).float())
        e = (d - d.amax(-1, keepdim=True)).exp()
        prob = (e / st.znuc.double()[:, None]).float().to(torch.bfloat16)
        assert torch.equal(st.greedy_tok.long(), (prob == prob.amax(-1, keepdim=True)).int().argmax(-1))
