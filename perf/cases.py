"""Performance cases of the paged-attention path: what an engine has the library do, one layer-call (or one
engine step of a few layers) at a time.

A case is a batch shape.  `chunks` sequences bring `chunk_lo`..`chunk_hi` new tokens over a prior context of
`prior_lo`..`prior_hi` cells (prefill chunks; a prior of 0 is a new prompt), then `decodes` sequences bring `n_q`
new tokens (1: decode, more: speculative verify) at a context of `ctx_lo`..`ctx_hi` cells.  The lengths are drawn
from `lens_seed`, so they belong to the case; block tables and values come from the seed.  `shared` leading cells
are one cached prefix of all chunks.

`entry` says how the call is made:
  fused   one launch that writes the step's K/V rows and attends (write_paged_attn)
  split   the K/V write, then attention (set_rows_kv, build_paged_attn)
  step    the engine runtime: one begin_step, then `layers` layers with RoPE (PagedAttnRuntime)
Calls are bound to their buffers once, as an engine that holds its arguments makes them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from iian_amd.paged_attn import (GGML_TYPE_F16, GGML_TYPE_F32, GGML_TYPE_Q8_0, KVPool, PagedAttnParams,
                                 PagedAttnRuntime, PagedBatch, RopeParams, bind_paged_attn, bind_set_rows_kv,
                                 bind_write_paged_attn, new_workspace)

BS = 16                       # the engine's block size
TYPES = {"f32": GGML_TYPE_F32, "f16": GGML_TYPE_F16, "q8_0": GGML_TYPE_Q8_0}
ELEM_BYTES = {"f32": 4.0, "f16": 2.0, "q8_0": 34.0 / 32.0}
FREQ_BASE = 1e6


def _case(name, entry, kv, H, Hkv, D, **kw):
    c = dict(name=name, entry=entry, kv=kv, H=H, Hkv=Hkv, D=D, chunks=0, chunk_lo=0, chunk_hi=0, prior_lo=0,
             prior_hi=0, shared=0, decodes=0, n_q=1, ctx_lo=0, ctx_hi=0, n_swa=0, softcap=0.0, layers=1, lens_seed=1)
    c.update(kw)
    return c


def listed():
    return [
        # a small model answering a few users: launches and latency
        _case("decode_small", "fused", "f16", 14, 2, 64, decodes=8, ctx_lo=64, ctx_hi=1024, lens_seed=1),
        # the headline: an 8B model's decode step over ragged contexts
        _case("decode_batch", "fused", "f16", 32, 8, 128, decodes=64, ctx_lo=512, ctx_hi=8192, lens_seed=2),
        # one or two users with a long document: few sequences, long contexts
        _case("decode_long", "fused", "f16", 32, 8, 128, decodes=2, ctx_lo=24000, ctx_hi=64000, lens_seed=3),
        # a sliding-window layer of a model with head size 256
        _case("decode_window", "fused", "f16", 16, 8, 256, decodes=32, ctx_lo=2048, ctx_hi=8192, n_swa=1024,
              lens_seed=4),
        # new prompts, no prior context
        _case("prefill_new", "split", "f16", 32, 8, 128, chunks=3, chunk_lo=700, chunk_hi=3000, lens_seed=5),
        # a global layer of a model with head size 256: prompt chunks over long contexts
        _case("prefill_d256", "split", "f16", 16, 8, 256, chunks=8, chunk_lo=256, chunk_hi=256, prior_lo=4096,
              prior_hi=16384, lens_seed=6),
        # an engine step: prompt chunks over a cached prefix beside running decodes
        _case("mixed_step", "step", "f16", 32, 8, 128, chunks=4, chunk_lo=400, chunk_hi=512, prior_lo=1024,
              prior_hi=4096, shared=1024, decodes=32, ctx_lo=1024, ctx_hi=4096, layers=2, lens_seed=7),
        # quantised KV: speculative verify of 5 tokens for a full batch
        _case("verify_q8", "split", "q8_0", 32, 8, 128, decodes=128, n_q=5, ctx_lo=4101, ctx_hi=4101, lens_seed=8),
        # quantised KV: an engine step with prompt chunks and decodes
        _case("mixed_q8", "step", "q8_0", 32, 8, 128, chunks=2, chunk_lo=300, chunk_hi=512, prior_lo=512,
              prior_hi=3072, decodes=24, ctx_lo=512, ctx_hi=4096, layers=2, lens_seed=9),
        # full-precision KV: decode
        _case("decode_f32", "split", "f32", 32, 8, 128, decodes=32, ctx_lo=512, ctx_hi=8192, lens_seed=10),
        # full-precision KV: an engine step with prompt chunks and decodes
        _case("mixed_f32", "step", "f32", 32, 8, 128, chunks=2, chunk_lo=200, chunk_hi=512, prior_lo=256,
              prior_hi=2048, decodes=16, ctx_lo=512, ctx_hi=4096, layers=1, lens_seed=11),
        # a head size off the powers of two, multi-head attention: chunks and decodes
        _case("mixed_d80", "split", "f16", 32, 32, 80, chunks=2, chunk_lo=200, chunk_hi=512, prior_lo=0,
              prior_hi=2048, decodes=16, ctx_lo=256, ctx_hi=4096, lens_seed=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges: fewer or as many sequences, other lengths and head layouts."""
    c = dict(rng.choice(listed()))
    name = c.pop("name")
    c["lens_seed"] = rng.randrange(1 << 30)
    if c["kv"] == "f16" and c["D"] == 128:
        c["H"], c["Hkv"], c["D"] = rng.choice([(32, 8, 128), (28, 4, 128), (32, 32, 96), (32, 8, 64), (14, 2, 64),
                                               (40, 8, 128), (9, 3, 64)])
    elif c["kv"] == "q8_0":
        c["H"], c["Hkv"], c["D"] = rng.choice([(32, 8, 128), (28, 4, 128), (32, 8, 64), (16, 8, 128), (14, 2, 64)])
    elif c["kv"] == "f32":
        c["H"], c["Hkv"], c["D"] = rng.choice([(32, 8, 128), (14, 2, 64), (32, 8, 64), (28, 4, 128), (16, 16, 96)])
    elif name == "mixed_d80":
        c["H"], c["Hkv"], c["D"] = rng.choice([(32, 32, 80), (20, 20, 80), (32, 8, 80), (32, 8, 112), (16, 2, 72)])
    if c["decodes"]:
        c["decodes"] = _log_int(rng, 1, c["decodes"])
        if name != "decode_long":
            hi = c["ctx_hi"]
            c["ctx_hi"] = _log_int(rng, max(64, hi // 8), hi)
            c["ctx_lo"] = _log_int(rng, 32, c["ctx_hi"])
        if c["entry"] != "step" and not c["chunks"] and c["H"] // c["Hkv"] <= 4:
            c["n_q"] = rng.choice([1, 1, 1, 2, 3, 5] if c["kv"] != "q8_0" else [1, 1, 2, 4, 5])
            c["ctx_lo"] = max(c["ctx_lo"], c["n_q"])
            c["ctx_hi"] = max(c["ctx_hi"], c["n_q"])
    if c["chunks"]:
        c["chunks"] = rng.randint(1, c["chunks"])
        c["chunk_hi"] = _log_int(rng, 33, c["chunk_hi"])
        c["chunk_lo"] = _log_int(rng, 17, c["chunk_hi"])
        if c["prior_hi"]:
            c["prior_hi"] = _log_int(rng, 64, c["prior_hi"])
            c["prior_lo"] = rng.randint(0, c["prior_hi"])
        c["shared"] = min(c["shared"], c["prior_lo"] // BS * BS)
    if name == "decode_window":
        c["n_swa"] = rng.choice([256, 512, 1024])
    if c["D"] in (64, 128, 256) and not c["n_swa"] and rng.random() < 0.15:
        c["softcap"] = 50.0
    return c


# ---- the batch of a case ----

def _lens(c):
    """(prior, new) cells of every sequence, in batch order."""
    r = np.random.default_rng(c["lens_seed"])
    prior = [int(r.integers(c["prior_lo"], c["prior_hi"] + 1)) for _ in range(c["chunks"])]
    new = [int(r.integers(c["chunk_lo"], c["chunk_hi"] + 1)) for _ in range(c["chunks"])]
    for _ in range(c["decodes"]):
        L = int(math.exp(r.uniform(math.log(c["ctx_lo"]), math.log(c["ctx_hi"])))) if c["ctx_lo"] < c["ctx_hi"] \
            else c["ctx_lo"]
        L = min(max(L, c["n_q"]), c["ctx_hi"])
        prior.append(L - c["n_q"])
        new.append(c["n_q"])
    return np.array(prior, np.int64), np.array(new, np.int64)


def work(case):
    c = case
    prior, new = _lens(c)
    H, Hkv, D, e = c["H"], c["Hkv"], c["D"], ELEM_BYTES[c["kv"]]
    T = int(new.sum())
    kv = pairs = 0
    for P, n in zip(prior.tolist(), new.tolist()):
        lo = max(0, P - c["n_swa"] + 1) if c["n_swa"] else 0
        kv += P + n - lo
        q = np.arange(P, P + n, dtype=np.int64)
        pairs += int((q + 1 - (np.maximum(0, q - c["n_swa"] + 1) if c["n_swa"] else 0)).sum())
    kv -= max(0, c["chunks"] - 1) * c["shared"]
    b = kv * Hkv * 2 * D * e                              # K and V of every attended cell
    b += T * H * D * 4 * 2                                # q in, attention out
    b += T * Hkv * D * 2 * 4                              # new K/V rows in (their stored copies are among kv)
    if c["entry"] == "step":
        b += T * H * D * 4                                # rotated q out
    b += int(((prior + new + BS - 1) // BS).sum()) * 4 + T * 12
    return {"bytes": float(b * c["layers"]), "flops": float(4 * H * D * pairs * c["layers"])}


def tolerance(case):
    # about four times the distance from exact(): 6.5e-7 where fp32 is kept throughout; 2.8e-4 at most with P
    # (and a Q8_0 V) rounded to f16, as the f16 matrix path does
    if case["kv"] == "f32" or case["D"] not in (64, 96, 128, 256):
        return {"rel": 4e-6, "max": 2e-4}
    return {"rel": 1.2e-3, "max": 5e-2}


def _inputs(c, seed):
    """Plain tensors of the case: block tables, the pools' bytes before the step, q and the new rows, per layer."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + 17)
    rng = np.random.default_rng(seed + 1)
    prior, new = _lens(c)
    S, T, n_embd = len(new), int(new.sum()), c["Hkv"] * c["D"]
    nblk = (prior + new + BS - 1) // BS
    sh = c["shared"] // BS
    num_blocks = int(nblk.sum()) + int(nblk.sum()) // 8 + 8
    perm = rng.permutation(num_blocks).astype(np.int32)
    ids, cur = [], sh
    for s in range(S):
        own = perm[cur:cur + int(nblk[s])].copy()
        cur += int(nblk[s])
        if s < c["chunks"]:
            own[:sh] = perm[:sh]
        ids.append(own)
    pos = np.concatenate([np.arange(p, p + n) for p, n in zip(prior, new)])
    seq = np.repeat(np.arange(S), new)
    cells = [own[np.arange(L) // BS].astype(np.int64) * BS + np.arange(L) % BS
             for own, L in zip(ids, (prior + new).tolist())]
    slots = np.concatenate([cl[int(p):] for cl, p in zip(cells, prior)])
    n_cells = num_blocks * BS

    def pool():
        if c["kv"] == "q8_0":   # blocks of a f16 scale and 32 quants of a normal value's spread
            b = torch.empty((n_cells, n_embd // 32, 34), dtype=torch.uint8, device="cuda")
            d = (torch.rand((n_cells, n_embd // 32, 1), generator=gen, device="cuda") * 0.01 + 0.012).half()
            b[:, :, :2] = d.view(torch.uint8)
            qs = torch.randn((n_cells, n_embd // 32, 32), generator=gen, device="cuda") * 55.0
            b[:, :, 2:] = qs.round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
            return b.view(n_cells, -1)
        x = torch.randn((n_cells, n_embd), generator=gen, device="cuda")
        return (x.half() if c["kv"] == "f16" else x).view(torch.uint8)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    layers = [dict(k_pool=pool(), v_pool=pool(), q=rand(T, c["H"], c["D"]) * 2.0, k_new=rand(T, n_embd),
                   v_new=rand(T, n_embd)) for _ in range(c["layers"])]
    return dict(prior=prior, new=new, ids=ids, pos=pos, seq=seq, slots=slots, cells=cells, layers=layers,
                num_blocks=num_blocks)


def prepare(case, seed):
    c = case
    x = _inputs(c, seed)
    S, T, max_q = len(x["new"]), len(x["pos"]), int(x["new"].max())
    n_embd, kv = c["Hkv"] * c["D"], TYPES[c["kv"]]
    max_blocks = max(len(i) for i in x["ids"])
    prm = PagedAttnParams(scale=1.0 / math.sqrt(c["D"]), softcap=c["softcap"], causal=True, n_swa=c["n_swa"])
    for ly in x["layers"]:
        ly["kp"], ly["vp"] = KVPool.wrap(ly["k_pool"], n_embd, kv), KVPool.wrap(ly["v_pool"], n_embd, kv)
        ly["out"] = torch.empty((T, c["H"], c["D"]), device="cuda")
    st = dict(entry=c["entry"], layers=x["layers"])
    if c["entry"] == "step":
        st["rt"] = PagedAttnRuntime(S, T, max_blocks, sum(len(i) for i in x["ids"]), c["H"], c["Hkv"], c["D"],
                                    c["D"], BS, x["num_blocks"], kv, kv)
        st["step"] = (x["ids"], x["prior"].astype(np.int32), x["new"].astype(np.int32))
        st["rope"] = RopeParams(n_dims=c["D"], mode=2, freq_base=FREQ_BASE)
        st["prm"] = prm
        for ly in x["layers"]:
            ly["q_rot"] = torch.empty_like(ly["q"])
        return st
    bt = np.zeros((S, max_blocks), np.int32)
    for s, own in enumerate(x["ids"]):
        bt[s, :len(own)] = own
    t = lambda a, dt: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda")  # noqa: E731
    batch = PagedBatch(block_tables=t(bt, torch.int32), seq_lens=t(x["prior"] + x["new"], torch.int32),
                       query_start_loc=t(np.concatenate([[0], np.cumsum(x["new"])]), torch.int32),
                       pos=t(x["pos"], torch.int32), slots=t(x["slots"], torch.int64), max_query_len=max_q,
                       block_size=BS)
    st["keep"] = batch, new_workspace(T, S, c["H"], c["Hkv"], c["D"], max_blocks, BS)
    ws, ly = st["keep"][1], x["layers"][0]
    if c["entry"] == "fused":
        st["calls"] = [bind_write_paged_attn(ly["q"], ly["k_new"], ly["v_new"], ly["kp"], ly["vp"], c["Hkv"], prm,
                                             batch, ly["out"], ws)]
    else:
        st["calls"] = [bind_set_rows_kv(ly["kp"], ly["vp"], ly["k_new"], ly["v_new"], batch.slots),
                       bind_paged_attn(ly["q"], ly["kp"], ly["vp"], c["Hkv"], prm, batch, ly["out"], ws)]
    return st


def run(state):
    if state["entry"] == "step":
        rt = state["rt"]
        rt.begin_step(*state["step"])
        for ly in state["layers"]:
            rt.layer(ly["q"], ly["k_new"], ly["v_new"], ly["kp"], ly["vp"], state["prm"], ly["out"],
                     rope=state["rope"], q_rot=ly["q_rot"])
    else:
        for call in state["calls"]:
            call()
    return [{k: ly[k] for k in ("out", "q_rot", "k_pool", "v_pool") if k in ly} for ly in state["layers"]]


# ---- the same in 64 bits ----

def _rope64(x, pos, n_head, D):
    """NEOX rotation in 64 bits of the angles the operator defines: an fp32 product chain over the pairs."""
    th = pos.astype(np.float32)
    scale = np.float32(FREQ_BASE) ** np.float32(-2.0 / D)
    angles = np.empty((len(pos), D // 2), np.float32)
    for j in range(D // 2):
        angles[:, j] = th
        th = th * scale
    a = torch.as_tensor(angles, device="cuda").double()[:, None, :]
    y = x.double().view(len(pos), n_head, D)
    y0, y1 = y[..., :D // 2], y[..., D // 2:]
    return torch.cat([y0 * a.cos() - y1 * a.sin(), y0 * a.sin() + y1 * a.cos()], -1)


def _stored64(rows, kv):
    """The values a pool row holds after the write of f32 rows."""
    if kv == "f32":
        return rows.float().double()
    if kv == "f16":
        return rows.float().half().double()
    v = rows.float().view(rows.shape[0], -1, 32)
    amax = v.abs().amax(-1, keepdim=True)
    d, inv = amax / 127.0, torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    return ((v * inv).round().clamp(-128, 127).double() * d.half().double()).view(rows.shape)


def _pool64(bytes_, kv):
    if kv == "f32":
        return bytes_.contiguous().view(torch.float32).double()
    if kv == "f16":
        return bytes_.contiguous().view(torch.float16).double()
    b = bytes_.view(bytes_.shape[0], -1, 34)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    return (b[:, :, 2:].contiguous().view(torch.int8).double() * d).view(bytes_.shape[0], -1)


def exact(case, seed):
    c = case
    x = _inputs(c, seed)
    H, Hkv, D, kv = c["H"], c["Hkv"], c["D"], c["kv"]
    gqa = H // Hkv
    res = []
    for ly in x["layers"]:
        r = dict(k_pool=None, v_pool=None)
        q, k_new = ly["q"].double(), ly["k_new"]
        if c["entry"] == "step":
            q = r["q_rot"] = _rope64(ly["q"], x["pos"], H, D)
            k_new = _rope64(k_new, x["pos"], Hkv, D).reshape(len(x["pos"]), -1)
            q = q.float().double()   # the rotated q is an f32 tensor
        out = torch.zeros((len(x["pos"]), H, D), dtype=torch.float64, device="cuda")
        t0 = 0
        for s, cl in enumerate(x["cells"]):
            P, n = int(x["prior"][s]), int(x["new"][s])
            lo = max(0, P - c["n_swa"] + 1) if c["n_swa"] else 0
            at = torch.as_tensor(cl[lo:P], device="cuda")
            K = torch.cat([_pool64(ly["k_pool"][at], kv), _stored64(k_new[t0:t0 + n], kv)]).view(-1, Hkv, D)
            V = torch.cat([_pool64(ly["v_pool"][at], kv), _stored64(ly["v_new"][t0:t0 + n], kv)]).view(-1, Hkv, D)
            cell = torch.arange(lo, P + n, device="cuda")[None, None, :]
            row = torch.arange(P, P + n, device="cuda")[:, None, None]
            hidden = cell > row
            if c["n_swa"]:
                hidden = hidden | (row - cell >= c["n_swa"])
            for h in range(Hkv):
                qh = q[t0:t0 + n, h * gqa:(h + 1) * gqa]
                sc = (qh.reshape(n * gqa, D) @ K[:, h].t().contiguous()) / math.sqrt(D)
                if c["softcap"]:
                    sc = c["softcap"] * torch.tanh(sc / c["softcap"])
                sc = sc.view(n, gqa, -1).masked_fill_(hidden, -math.inf)
                p = torch.softmax(sc, -1).view(n * gqa, -1)
                out[t0:t0 + n, h * gqa:(h + 1) * gqa] = (p @ V[:, h].contiguous()).view(n, gqa, D)
            t0 += n
        r["out"] = out
        res.append(r)
    return res
