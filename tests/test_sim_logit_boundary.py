"""The greedy statistics' nucleus cut on rows whose probability mass ends at a rounding
boundary: the sums that the finish kernel's scan gives the empty 64-key stretches after
the last token differ by an ulp and lie on both sides of top_p, so several threads, of
stretches without tokens, pass the crossing test.  sf_logits.hip's own source runs on
the CPU simulator, compiled to trap on any array index outside its array."""

import ctypes
import subprocess
import sys

import numpy as np
import pytest
import torch

if __name__ == "__main__":
    sys.path.insert(0, sys.argv[1])

from tests.simlib import CSRC, FLAGS, ROOT, SIM, compiler

V = 152064
F = np.float32
BITS = np.arange(65536)
KEY = np.where(BITS & 0x8000, ~BITS & 0xffff, BITS | 0x8000)   # order key of a bf16 pattern
VAL = np.empty(65536, F)                                       # value of a key
VAL[KEY] = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).float()


def bf16(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=F)).to(torch.bfloat16)


def scan(x):
    """The kernel's inclusive prefix sums of 1024 fp32 terms: a shuffle scan per 64, then
    the totals of the 64s in order."""
    v = x.reshape(16, 64).copy()
    for o in (1, 2, 4, 8, 16, 32):
        n = v.copy()
        n[:, o:] = v[:, o:] + v[:, :-o]
        v = n
    base, inc = F(0), np.empty((16, 64), F)
    for w in range(16):
        inc[w] = base + v[w]
        base = F(base + v[w, 63])
    return inc.reshape(-1)


def stretch_sums(cnt):
    """(Z, per-stretch bf16 probability mass) from the counts of every key."""
    keys = np.nonzero(cnt)[0][::-1]
    e = np.exp(VAL[keys] - VAL[keys[0]])

    def parts(term):
        out = np.zeros(1024, F)
        for k, x in zip(keys, term):
            out[(65535 - k) // 64] += F(cnt[k]) * x
        return out
    z = scan(parts(e))[-1]
    return z, parts(bf16(e / z).float().numpy())


def boundary_row(seed):
    """(logits [V] bf16, top_p): a row of normal logits without values near zero (so
    that the stretches below the smallest positive value are empty), tokens moved
    between its values until the positive mass straddles a rounding boundary, top_p."""
    rng = np.random.default_rng(seed)
    while True:
        x = rng.normal(0, 1, V) * rng.uniform(.8, 1.6) + rng.uniform(-1.2, -.2)
        x = bf16(np.where(np.abs(x) < 0.02, -0.5, x)).view(torch.int16).numpy()
        cnt = np.bincount(KEY[x.astype(np.int64) & 0xffff], minlength=65536)
        for _ in range(40):
            z, mass = stretch_sums(cnt)
            empty = scan(mass)[np.nonzero(mass[:512])[0].max():512]
            m = float(np.median(empty))
            if not .125 <= m < 1:
                break
            steps = 256 if m >= .5 else 512 if m >= .25 else 1024   # bf16 steps per 1.0 at m
            mid = (np.floor(m * steps) + .5) / steps
            r = bf16(empty).float().numpy()
            if r.min() < mid < r.max():
                return bf16(VAL[np.repeat(np.arange(65536), cnt)][rng.permutation(V)]), mid
            pos = np.nonzero(cnt[32768:] > 3)[0] + 32768
            pos = pos[VAL[pos] < VAL[np.nonzero(cnt)[0].max()] - .5]
            neg = np.nonzero(cnt[:32768] > 3)[0]
            p = bf16(np.exp(VAL[pos] - VAL[np.nonzero(cnt)[0].max()]) / z).double().numpy()
            diff = mid - m
            if abs(diff) > 4 * p.max():      # tokens between the signs
                for _ in range(min(int(abs(diff) / np.median(p)) + 1, 3000)):
                    a, b = rng.choice(pos), rng.choice(neg)
                    a, b = (b, a) if diff > 0 else (a, b)
                    if cnt[a] > 1:
                        cnt[a] -= 1
                        cnt[b] += 1
            else:                            # a token between two positive values
                i, j = rng.integers(0, len(pos), (2, 4000))
                k = np.argmin(np.abs(p[j] - p[i] - diff) + (cnt[pos[i]] < 2))
                cnt[pos[i[k]]] -= 1
                cnt[pos[j[k]]] += 1


def _child(lib_path, data):
    lib = ctypes.CDLL(lib_path)
    lib.sf_logit_stats_workspace_bytes.restype = ctypes.c_size_t
    d = torch.load(data, weights_only=True)
    out = []
    for x, top_p in zip(d["rows"], d["top_p"]):
        ws = torch.zeros(lib.sf_logit_stats_workspace_bytes(1), dtype=torch.uint8)
        o = {k: torch.zeros(8, dtype=t) for k, t in (
            ("top_idx", torch.int32), ("top_val", torch.float32), ("zfull", torch.float32),
            ("znuc", torch.float32), ("greedy", torch.int32), ("conf", torch.float32),
            ("conf_full", torch.float32))}
        st = lib.sf_logit_stats(ctypes.c_void_p(x.data_ptr()), 1, V, ctypes.c_longlong(V),
                                ctypes.c_float(top_p),
                                *(ctypes.c_void_p(t.data_ptr()) for t in o.values()),
                                ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(ws.numel()), None)
        assert st == 0 and int(ws[:65536 * 4].count_nonzero()) == 0
        out.append({k: t[:1].clone() for k, t in o.items()})
    torch.save(out, data + ".out")


def test_cut_at_an_empty_stretch(tmp_path):
    from tests.test_gpu_logit_stats import nucleus_mass64, reference_greedy, ulp_bf16
    cxx = compiler()
    if cxx is None:
        pytest.skip("no clang++ (the simulator needs clang's vector extensions)")
    for f in ("sf_logits.hip", "sf_index.h"):
        (tmp_path / f).write_text((CSRC / f).read_text())
    lib = tmp_path / "logits.so"
    r = subprocess.run([cxx, *FLAGS, "-fsanitize=bounds", "-fsanitize-trap=bounds", f"-I{SIM}",
                        f"-I{ROOT / 'include'}", f"-I{CSRC}", "-x", "c++", "-shared",
                        str(tmp_path / "sf_logits.hip"), "-o", str(lib), "-lpthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    rows, top_p = zip(*(boundary_row(s) for s in (1, 2, 3, 4)))
    data = str(tmp_path / "rows.pt")
    torch.save(dict(rows=torch.stack(rows), top_p=list(map(float, top_p))), data)
    r = subprocess.run([sys.executable, __file__, str(ROOT), str(lib), data],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, (r.returncode, r.stderr[-3000:])
    for x, p, got in zip(rows, top_p, torch.load(data + ".out", weights_only=True)):
        x = x[None]
        zn64, z64 = nucleus_mass64(x, float(p))
        # the cut moves by one token (e <= 1) where the mass rounds across top_p
        assert float((got["znuc"].double() - zn64).abs()) <= 1e-5 * float(z64) + 1.0
        tok, conf = reference_greedy(x, float(p))
        assert float((got["conf"] - conf.float()).abs()) <= float(ulp_bf16(conf))
        if float(got["conf"]) == float(conf):
            assert int(got["greedy"]) == int(tok)


if __name__ == "__main__":
    _child(sys.argv[2], sys.argv[3])
