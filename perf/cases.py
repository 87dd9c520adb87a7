"""Performance cases of the tiered-KV attention path, each through a public entry point.

A case is a dict of plain values; ``kind`` names the entry point:

  decode   one decode token over a list of device chunks (``triton_chunked_attention``)
  tiered   one decode step of a layer that picks its cold chunks (``TieredDecodeLayer``)
  ragged   the same for a batch of sequences of different lengths (``RaggedTieredDecodeLayer``)
  kivi     one decode step over a 2-bit cold tier and recent rows (``KiviDecodeLayer``)
  cache    one decode step of the Path-D cache, cold chunks in pinned host memory (``HALOCacheChunked``)
  prefill  a block of query rows over prior chunks and its own rows (``prefill_attention``)
  store    quantise-on-demote and the dequantised copy (``kivi.quantize`` / ``kivi.dequantize``)
  means    mean-key page scoring at a peel (``chunk_means`` / ``score_topk``)
  quest    bounding-box page scoring at a peel (``page_minmax`` / ``quest_score_topk``)

Keys and values are N(0, 1); where chunks are selected, four key channels
have standard deviation 8, as the high-variance channels of real keys do.
"""
from __future__ import annotations

import math
import random

import torch

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ESIZE = {"bf16": 2, "f16": 2, "f32": 4}
GROUP = 32  # tokens of a KIVI block
DEV = "cuda"


def listed():
    return [
        # the smallest call: one layer of a short chat turn, where launches count
        dict(name="decode_4k", kind="decode", B=1, H=32, H_kv=8, D=128, T=4096, chunk=1024, dtype="bf16"),
        # one layer of the 32k-context headline workload: 8 hot chunks and the top 4 of 24 cold ones
        dict(name="tiered_32k", kind="tiered", B=1, H=32, H_kv=8, D=128, chunk=1024, n_hot=8, n_cold=24, top_k=4,
             dtype="bf16"),
        # a serving batch of 16 sequences of 8k to 128k tokens, each picking its own cold chunks
        dict(name="ragged_16x", kind="ragged", B=16, H=32, H_kv=8, D=128, lo=8192, hi=131072, ctx_seed=3, chunk=2048,
             top_k=8, dtype="bf16"),
        # one layer of a 28/4-head model at 128k context with everything but the recent rows in 2 bits
        dict(name="kivi_128k", kind="kivi", B=1, H=28, H_kv=4, D=128, T=131072, recent=128, dtype="f16"),
        # what a wrapped model's layer calls for each token: 512 rows on the GPU, the rest in pinned host chunks
        dict(name="cache_8k", kind="cache", B=1, H=32, H_kv=8, D=128, T=8192, chunk=1024, recent=512, dtype="bf16"),
        # the last slice of a long prompt: 4096 rows over 28k prior ones
        dict(name="prefill_long", kind="prefill", B=1, H=32, H_kv=8, D=128, T_q=4096, prior=28672, chunk=1024,
             dtype="bf16", lse=False),
        # a small slice of a chunked prefill in the middle of a prompt
        dict(name="prefill_slice", kind="prefill", B=1, H=32, H_kv=8, D=128, T_q=512, prior=8192, chunk=1024,
             dtype="bf16", lse=False),
        # the last, ragged slice of a prompt, with head dim 64, partials to be merged
        dict(name="prefill_tail", kind="prefill", B=2, H=16, H_kv=4, D=64, T_q=137, prior=3000, chunk=512,
             dtype="f16", lse=True),
        # a prompt of an fp32 model
        dict(name="prefill_f32", kind="prefill", B=1, H=16, H_kv=4, D=64, T_q=512, prior=1536, chunk=512,
             dtype="f32", lse=False),
        # a 32k prompt demoted to the 2-bit tier and handed back dequantised
        dict(name="store_32k", kind="store", B=1, H_kv=8, D=128, T=32768, bits=2, dtype="bf16"),
        # placement at a peel, mean-key scorer with its default 16-row pages
        dict(name="means_8k", kind="means", B=1, H=32, H_kv=8, D=128, T=8192, page=16, ratio=4, dtype="bf16"),
        # placement at a peel, bounding-box scorer over the last query block
        dict(name="quest_32k", kind="quest", B=1, H=32, H_kv=8, D=128, T_q=1, T=32768, page=16, ratio=4, dtype="bf16"),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "tiered", "ragged", "kivi", "cache", "prefill", "prefill", "prefill", "store", "means",
                       "quest"])
    H, H_kv = rng.choice([(32, 8), (28, 4), (16, 4), (8, 8)])
    D = rng.choice([64, 128, 128])
    c = dict(kind=kind, B=1, H=H, H_kv=H_kv, D=D, dtype=rng.choice(["bf16", "bf16", "f16"]))
    if kind == "decode":
        c["dtype"] = rng.choice(["bf16", "f16", "f32"])
        c.update(B=rng.choice([1, 1, 2, 4]), T=_log(rng, 300, 32768), chunk=rng.choice([256, 512, 1024, 2048]))
    elif kind == "tiered":
        n = _log(rng, 8, 64)
        c.update(chunk=rng.choice([256, 512, 1024]), n_hot=max(1, n // 4), n_cold=n - max(1, n // 4),
                 top_k=rng.randint(2, 6))
    elif kind == "ragged":
        c.update(B=rng.randint(2, 12), lo=8192, hi=_log(rng, 16384, 98304), ctx_seed=rng.randrange(1000), chunk=2048,
                 top_k=rng.randint(2, 8))
    elif kind == "kivi":
        c.update(T=32 * _log(rng, 64, 4096) + rng.randint(0, 31), recent=rng.choice([32, 128]))
    elif kind == "cache":
        c.update(T=_log(rng, 2100, 8192), chunk=rng.choice([512, 1024]), recent=rng.choice([64, 512]))
    elif kind == "prefill":
        c["dtype"] = rng.choice(["bf16", "bf16", "f16", "f32"])
        f32 = c["dtype"] == "f32"
        c.update(B=rng.choice([1, 1, 2]), T_q=_log(rng, 8, 512 if f32 else 2048),
                 prior=rng.choice([0, _log(rng, 64, 2048 if f32 else 16384)]), chunk=rng.choice([512, 1024]),
                 lse=rng.choice([False, True]))
    elif kind == "store":
        c.update(T=32 * _log(rng, 4, 1024), bits=rng.choice([2, 2, 4, 8]))
    elif kind == "means":
        c.update(T=_log(rng, 1024, 16384), page=rng.choice([16, 32]), ratio=rng.choice([2, 4, 8]))
    else:
        c.update(T_q=rng.choice([1, 1, 4]), T=_log(rng, 1024, 65536), page=rng.choice([16, 32]),
                 ratio=rng.choice([2, 4, 8]))
    return c


# ---------------------------------------------------------------- shapes

def _cuts(T: int, chunk: int):
    return [(s, min(chunk, T - s)) for s in range(0, T, chunk)]


def _contexts(case):
    r = random.Random(case["ctx_seed"])
    ch = case["chunk"]
    return [max(ch, int(r.uniform(case["lo"], case["hi"])) // ch * ch) for _ in range(case["B"])]


def _hot_cold(T: int, chunk: int):
    n = T // chunk
    hot = max(1, n // 4)
    return n - hot, hot  # cold chunks come first


def _pages(case):
    P = case["T"] // case["page"]
    return P, min(P, max(4, (P + case["ratio"] - 1) // case["ratio"]))


def _kivi_split(case):
    """(quantised rows, recent rows): whole blocks of all but the recent window."""
    n = max(0, case["T"] - case["recent"]) // GROUP * GROUP
    return n, case["T"] - n


# ---------------------------------------------------------------- inputs

def _randn(gen, shape, dtype, sigma=None):
    x = torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32)
    if sigma is not None:
        x.mul_(sigma)
    return x.to(dtype)


def _gen(seed: int):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _planted(gen, D: int):
    s = torch.ones(D, device=DEV)
    s[torch.randperm(D, generator=gen, device=DEV)[:4]] = 8.0
    return s


def _inputs(case, seed: int):
    """q, k, v (and for ragged cases lists of k, v) from the seed alone."""
    g, dt, kind = _gen(seed), DTYPES[case["dtype"]], case["kind"]
    B, D, H_kv = case["B"], case["D"], case["H_kv"]
    if kind == "ragged":
        s = _planted(g, D)
        q = _randn(g, (B, case["H"], D), dt)
        ks, vs = [], []
        for T in _contexts(case):
            ks.append(_randn(g, (H_kv, T, D), dt, s))
            vs.append(_randn(g, (H_kv, T, D), dt))
        return q, ks, vs
    if kind == "tiered":
        s = _planted(g, D)
        T = (case["n_hot"] + case["n_cold"]) * case["chunk"]
        return (_randn(g, (B, case["H"], D), dt), _randn(g, (B, H_kv, T, D), dt, s), _randn(g, (B, H_kv, T, D), dt))
    if kind in ("means", "quest"):
        return (_randn(g, (B, case["H"], case.get("T_q", 1), D), dt),
                _randn(g, (B, H_kv, case["T"], D), dt, _planted(g, D)), None)
    if kind == "store":
        return None, _randn(g, (B, H_kv, case["T"], D), dt), _randn(g, (B, H_kv, case["T"], D), dt)
    T_q = case.get("T_q", 1)
    T = case["prior"] + T_q if kind == "prefill" else case["T"]
    return (_randn(g, (B, case["H"], T_q, D), dt), _randn(g, (B, H_kv, T, D), dt), _randn(g, (B, H_kv, T, D), dt))


def prepare(case, seed):
    kind, B, D, H_kv = case["kind"], case["B"], case["D"], case["H_kv"]
    H, dt = case.get("H"), DTYPES[case["dtype"]]
    q, k, v = _inputs(case, seed)
    st = dict(case=case, q=q, k=k, v=v, scale=1.0 / math.sqrt(D))
    if kind == "decode":
        st["chunks"] = [(k[..., s:s + n, :], v[..., s:s + n, :], s, True) for s, n in _cuts(case["T"], case["chunk"])]
    elif kind == "tiered":
        from halo_amd.decode import ChunkRef
        from halo_amd.tiered import TieredDecodeLayer
        ch, n_cold = case["chunk"], case["n_cold"]
        refs = [ChunkRef(k[..., s:s + n, :], v[..., s:s + n, :], s, True) for s, n in _cuts(k.shape[2], ch)]
        st["layer"] = TieredDecodeLayer(B=B, H=H, H_kv=H_kv, D=D, dtype=dt, hot=refs[n_cold:], cold=refs[:n_cold],
                                        top_k=min(case["top_k"], n_cold), device=DEV)
        st["q_pos"] = torch.full((B,), k.shape[2] - 1, device=DEV, dtype=torch.int64)
    elif kind == "ragged":
        from halo_amd.decode import ChunkRef
        from halo_amd.tiered import RaggedTieredDecodeLayer
        rows, ch = [], case["chunk"]
        for b, (kb, vb) in enumerate(zip(k, v)):
            refs = [ChunkRef(kb[:, s:s + n], vb[:, s:s + n], s, True, batch=b) for s, n in _cuts(kb.shape[1], ch)]
            n_cold, _ = _hot_cold(kb.shape[1], ch)
            rows.append((refs[n_cold:], refs[:n_cold]))
        st["layer"] = RaggedTieredDecodeLayer(H=H, H_kv=H_kv, D=D, dtype=dt, rows=rows, top_k=case["top_k"], device=DEV)
        st["q_pos"] = torch.tensor([kb.shape[1] - 1 for kb in k], device=DEV, dtype=torch.int64)
    elif kind == "kivi":
        from halo_amd import kivi
        from halo_amd.decode import ChunkRef
        n, rec = _kivi_split(case)
        st["blocks"] = kivi.quantize(k[:, :, :n], v[:, :, :n])
        recent = [ChunkRef(k[:, :, n:].contiguous(), v[:, :, n:].contiguous(), n, True)] if rec else []
        st["layer"] = kivi.KiviDecodeLayer(B=B, H=H, H_kv=H_kv, D=D, dtype=dt, cold_blocks=st["blocks"], recent=recent,
                                           device=DEV)
        st["q_pos"] = torch.full((B,), case["T"] - 1, device=DEV, dtype=torch.int64)
        st["k"] = st["v"] = None
    elif kind == "cache":
        from halo_amd import HALOCacheChunked
        cache = HALOCacheChunked(chunk_size=case["chunk"], recent_window=case["recent"])
        T = case["T"]
        for s, n in _cuts(T - 1, 2048):
            cache.update(k[:, :, s:s + n], v[:, :, s:s + n], 0)
        cache.update(k[:, :, T - 1:], v[:, :, T - 1:], 0)  # the first decode token starts the peel
        st["cache"] = cache
    elif kind == "prefill":
        from halo_amd.decode import ChunkRef
        prior = case["prior"]
        st["chunks"] = [ChunkRef(k[..., s:s + n, :], v[..., s:s + n, :], s, False) for s, n in _cuts(prior, case["chunk"])]
        st["chunks"].append(ChunkRef(k[..., prior:, :], v[..., prior:, :], prior, True))
    elif kind == "means":
        st["elig"] = torch.arange(_pages(case)[0], device=DEV, dtype=torch.int32)
    return st


def run(st):
    case, q, k, v = st["case"], st["q"], st["k"], st["v"]
    kind, B, D = case["kind"], case["B"], case["D"]
    if kind == "decode":
        from halo_amd.triton_chunked import triton_chunked_attention
        out, lse = triton_chunked_attention(q, st["chunks"], scale=st["scale"], return_lse=True)
        return {"out": out, "lse": lse}
    if kind in ("tiered", "ragged", "kivi"):
        layer = st["layer"]
        q3 = q[:, :, 0] if q.dim() == 4 else q
        out = torch.empty((B, case["H"], D), device=DEV, dtype=q.dtype)
        lse = torch.empty((B, case["H"]), device=DEV, dtype=torch.float32)
        layer.step(q3, scale=st["scale"], out=out, lse=lse, q_pos=st["q_pos"])
        if kind == "kivi":
            return {"out": out, "lse": lse}
        return {"out": out, "lse": lse, "idx": layer.idx}
    if kind == "cache":
        out, lse = st["cache"].compute_attention(q, layer_idx=0, scaling=st["scale"], return_lse=True)
        return {"out": out, "lse": lse}
    if kind == "prefill":
        from halo_amd.prefill import prefill_attention
        res = prefill_attention(q, st["chunks"], scale=st["scale"], q_start=case["prior"], return_lse=case["lse"])
        return {"out": res[0], "lse": res[1]} if case["lse"] else {"out": res}
    if kind == "store":
        from halo_amd import kivi
        blocks = kivi.quantize(k, v, bits=case["bits"])
        kd, vd = kivi.dequantize(blocks, D=D, dtype=k.dtype, bits=case["bits"])
        return {"blocks": blocks, "k": kd, "v": vd}
    P, K = _pages(case)
    if kind == "means":
        from halo_amd.chunk_scorer import chunk_means, score_topk
        km = chunk_means(k, case["page"])
        idx, scores = score_topk(q, km, st["elig"], K, normalize=True, P_total=P)
        return {"means": km, "idx": idx, "scores": scores}
    from halo_amd.quest_scorer import page_minmax, quest_score_topk
    kmin, kmax = page_minmax(k, case["page"])
    idx, _, scores = quest_score_topk(q, kmin, kmax, K, want_scores=True)
    return {"kmin": kmin, "kmax": kmax, "idx": idx, "scores": scores}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind, e, B, D = case["kind"], ESIZE[case["dtype"]], case["B"], case["D"]
    H, H_kv = case.get("H", 0), case["H_kv"]
    qo = 2 * B * H * D * e + B * H * 4
    if kind in ("decode", "cache"):
        rows = B * case["T"]
        return {"bytes": 2 * rows * H_kv * D * e + qo, "flops": 4 * rows * H * D}
    if kind == "tiered":
        rows = B * (case["n_hot"] + min(case["top_k"], case["n_cold"])) * case["chunk"]
        return {"bytes": 2 * rows * H_kv * D * e + B * case["n_cold"] * H_kv * D * e + qo, "flops": 4 * rows * H * D}
    if kind == "ragged":
        rows = cold = 0
        for T in _contexts(case):
            n_cold, n_hot = _hot_cold(T, case["chunk"])
            rows += (n_hot + min(case["top_k"], n_cold)) * case["chunk"]
            cold += n_cold
        return {"bytes": 2 * rows * H_kv * D * e + cold * H_kv * D * e + qo, "flops": 4 * rows * H * D}
    if kind == "kivi":
        n, rec = _kivi_split(case)
        return {"bytes": B * H_kv * (n // GROUP * 24 * D + rec * 2 * D * e) + qo, "flops": 4 * B * (n + rec) * H * D}
    if kind == "prefill":
        T_q, prior = case["T_q"], case["prior"]
        seen = T_q * prior + T_q * (T_q + 1) // 2
        return {"bytes": 2 * B * (prior + T_q) * H_kv * D * e + 2 * B * H * T_q * D * e + (B * H * T_q * 4 if case["lse"] else 0),
                "flops": 4 * B * H * D * seen}
    rows = B * H_kv * case["T"]
    if kind == "store":
        blocks = rows // GROUP * (8 * case["bits"] * D + 8 * D)
        return {"bytes": 2 * rows * D * e + blocks + 2 * rows * D * e, "flops": 10 * rows * D}
    P, K = _pages(case)
    meta = (1 if kind == "means" else 2) * B * H_kv * P * D * e
    T_q = case.get("T_q", 1)
    return {"bytes": rows * D * e + meta + B * H * T_q * D * e + 4 * (K + P),
            "flops": rows * D + (2 if kind == "means" else 4) * B * H_kv * T_q * P * D}


def tolerance(case):
    """16-bit attention: the output is rounded to 8 (bf16) or 11 (f16) bits and
    the probabilities to the same in front of the second product.  Measured
    against ``exact``, of which this is about four times: 2.3e-3 in bf16,
    2.9e-4 in f16 (1.2e-3 over 2-bit blocks, whose zeros and scales enter the
    products in 11 bits), up to 1e-6 in f32 over the longest sums."""
    if case["kind"] in ("store", "quest", "means"):
        return "exact"  # fixed orders of summation: bytes, page means and ranks are pinned bit for bit
    if case["kind"] == "kivi" and case["dtype"] == "f16":
        return {"rel": 5e-3}
    return {"rel": {"bf16": 1e-2, "f16": 1.5e-3, "f32": 5e-6}[case["dtype"]]}


# ---------------------------------------------------------------- the same in 64 bits

def _attend(q, k, v, scale, q0=None):
    """q (H, T_q, D) over k, v (H_kv, T, D) in 64 bits; query row i sees keys up to q0 + i (None: all)."""
    H, T_q, D = q.shape
    rep = H // k.shape[0]
    T = k.shape[1]
    out = torch.empty((H, T_q, D), device=q.device, dtype=torch.float64)
    lse = torch.empty((H, T_q), device=q.device, dtype=torch.float64)
    step = max(1, (1 << 27) // T)
    key = torch.arange(T, device=q.device)
    for h in range(H):
        kt, vh = k[h // rep].double().t().contiguous(), v[h // rep].double()
        for i in range(0, T_q, step):
            s = (q[h, i:i + step].double() @ kt) * scale
            if q0 is not None:
                pos = q0 + torch.arange(i, min(i + step, T_q), device=q.device)
                s.masked_fill_(key[None] > pos[:, None], float("-inf"))
            lse[h, i:i + step] = torch.logsumexp(s, dim=-1)
            out[h, i:i + step] = torch.softmax(s, dim=-1) @ vh
    return out, lse


def _batch(q, k, v, scale, q0=None):
    r = [_attend(q[b], k[b], v[b], scale, q0) for b in range(q.shape[0])]
    return torch.stack([x[0] for x in r]), torch.stack([x[1] for x in r])


def _round(x, dtype):
    return x.float().to(dtype).double()


def _mean_scores(q, kmean, dtype):
    """q (B, H, D), kmean (B, H_kv, P, D) 64-bit values of ``dtype`` -> (B, H_kv, P): the GQA-mean query, kept in the key dtype, against every page mean."""
    B, H, D = q.shape
    qg = _round(q.double().reshape(B, kmean.shape[1], -1, D).mean(2), dtype)
    return (kmean * qg[:, :, None]).sum(-1)


def _chunk_kmean(k, chunk, dtype):
    """Mean key of every ``chunk`` rows of k (..., T, D), kept in the key dtype."""
    T, D = k.shape[-2:]
    n = T // chunk
    return _round(k[..., :n * chunk, :].double().reshape(*k.shape[:-2], n, chunk, D).mean(-2), dtype)


def _picked(k, ids, chunk):
    return torch.cat([k[:, i * chunk:(i + 1) * chunk] for i in ids], dim=1)


def _kivi_values(x, bits, dim):
    """KIVI's affine codes of x, groups of 32 along ``dim``: (code, scale, zero), each elementary operation rounded to x's type."""
    qmax = (1 << bits) - 1
    g = x.movedim(dim, -1)
    g = g.reshape(*g.shape[:-1], -1, GROUP)
    lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
    scale = (hi - lo).clamp_min(1e-8) / qmax
    code = ((g - lo) / scale).nan_to_num(0.0).round().clamp(0, qmax)

    def back(t):
        t = t.expand_as(g)
        return t.reshape(*t.shape[:-2], -1).movedim(-1, dim)
    return back(code), back(scale), back(lo)


def exact(case, seed):
    kind, D = case["kind"], case["D"]
    scale = 1.0 / math.sqrt(D)
    dt = DTYPES[case["dtype"]]
    q, k, v = _inputs(case, seed)
    if kind in ("decode", "cache"):
        out, lse = _batch(q, k, v, scale)
        return {"out": out, "lse": lse if kind == "cache" else lse[:, :, 0]}
    if kind == "prefill":
        out, lse = _batch(q, k, v, scale, case["prior"])
        return {"out": out, "lse": lse} if case["lse"] else {"out": out}
    if kind == "tiered":
        ch, n_cold = case["chunk"], case["n_cold"]
        sc = _mean_scores(q, _chunk_kmean(k[:, :, :n_cold * ch], ch, dt), dt).amax((0, 1))
        ids = sc.topk(min(case["top_k"], n_cold)).indices.sort().values.tolist()
        ids += list(range(n_cold, n_cold + case["n_hot"]))
        r = [_attend(q[b, :, None], _picked(k[b], ids, ch), _picked(v[b], ids, ch), scale) for b in range(case["B"])]
        return {"out": torch.stack([x[0][:, 0] for x in r]), "lse": torch.stack([x[1][:, 0] for x in r]), "idx": None}
    if kind == "ragged":
        ch, r = case["chunk"], []
        for b, (kb, vb) in enumerate(zip(k, v)):
            n_cold, n_hot = _hot_cold(kb.shape[1], ch)
            ids = list(range(n_cold, n_cold + n_hot))
            if n_cold:
                sc = _mean_scores(q[b:b + 1], _chunk_kmean(kb[None, :, :n_cold * ch], ch, dt), dt).amax((0, 1))
                ids = sc.topk(min(case["top_k"], n_cold)).indices.sort().values.tolist() + ids
            r.append(_attend(q[b, :, None], _picked(kb, ids, ch), _picked(vb, ids, ch), scale))
        return {"out": torch.stack([x[0][:, 0] for x in r]), "lse": torch.stack([x[1][:, 0] for x in r]), "idx": None}
    if kind == "kivi":
        n, _ = _kivi_split(case)
        full = []
        for x, dim in ((k, -2), (v, -1)):
            code, sc, zero = _kivi_values(x[:, :, :n], 2, dim)
            full.append(torch.cat([code.double() * sc.double() + zero.double(), x[:, :, n:].double()], dim=2))
        out, lse = _batch(q, full[0], full[1], scale)
        return {"out": out[:, :, 0], "lse": lse[:, :, 0]}
    if kind == "store":
        back = []
        for x, dim in ((k, -2), (v, -1)):
            code, sc, zero = _kivi_values(x, case["bits"], dim)
            back.append(code.double() * sc.double() + zero.double())
        return {"blocks": None, "k": back[0], "v": back[1]}
    P, page = _pages(case)[0], case["page"]
    if kind == "means":
        km = k[:, :, :P * page].double().reshape(*k.shape[:2], P, page, D).mean(3)
        a = _mean_scores(q[:, :, -1], _round(km, dt), dt).amax((0, 1))
        a = a - a.min()
        return {"means": km, "idx": None, "scores": (a / a.max())[None]}
    kp = k[:, :, :P * page].double().reshape(*k.shape[:2], P, page, D)
    kmin, kmax = kp.amin(3), kp.amax(3)
    B, H, T_q, _ = q.shape
    qg = _round(q.double().reshape(B, case["H_kv"], -1, T_q, D).mean(2), dt)
    best = torch.full((P,), float("-inf"), device=q.device, dtype=torch.float64)
    for t in range(T_q):
        x = qg[:, :, t, None]
        best = torch.maximum(best, torch.maximum(x * kmin, x * kmax).sum(-1).amax((0, 1)))
    return {"kmin": kmin, "kmax": kmax, "idx": None, "scores": best[None]}
