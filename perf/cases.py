"""The performance cases: calls that programs make of this library, small to large.

Four ways in, as programs use them:

  step     hip.DeviceProblem + hip.launch_hip: a device-level caller (an engine with its own cache)
           keeps the problem's buffers and enqueues one certified attention step per pass
  forward  serving.ExactAttentionBackend.forward over a PagedKVCache: append the new tokens' K/V and
           attend, one layer of a serving loop. Each pass first cuts the slots back to their
           prefix, as a speculative loop does whose drafts were all rejected, so passes repeat
  hf       serving.hf_attention: the transformers attention function, which waits for its flags
  host     attention_hip on host arrays: one head's causal rows, as the fixture check calls it

Keys and values are standard normal bf16; long contexts have outlier key channels, as in the
long-context configuration. Outputs are certified: every correct implementation gives the same
bits, so every tolerance is "exact".
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

import exactattention_amd as ea
from exactattention_amd import configs, hip
from exactattention_amd.formats import default_alpha_bits
from exactattention_amd.serving import ExactAttentionBackend, PagedKVCache, hf_attention

# fields of a "step" case: B sequences of kv_min..kv keys (kv_min = kv: all equal; else spread over
# the logarithm by `lens`), T query tokens at the end of each sequence (tree: a draft tree of T nodes
# after the keys), Hq query heads on Hkv KV heads, head dim d, page (0: contiguous), out, digits (the
# K/V digit tiles kept across steps), outliers (4 key channels of 30 times the scale per KV head)
_STEP = dict(kind="step", T=1, d=128, page=16, out="bf16", tree=False, digits=False, outliers=False, lens=0)


def _step(name, **kw):
    c = dict(_STEP, **kw)
    c.setdefault("kv_min", c["kv"])
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one decode token of a short chat turn through transformers: latency and launches only
        dict(name="hf_decode_300", kind="hf", B=1, ql=1, kl=300, Hq=16, Hkv=8, d=128),
        # batched paged decode, the benchmark's headline shape (two query heads per KV head)
        _step("decode_gqa2_32x4k", B=32, kv=4096, Hq=16, Hkv=8),
        # batched paged decode of a wide-GQA model, lengths as a running batch has them
        _step("decode_gqa8_ragged", B=32, kv=4096, kv_min=512, lens=3, Hq=64, Hkv=8),
        # a small batch's decode through the serving layer: append and attend
        dict(name="forward_decode_5", kind="forward", B=5, tok=1, last=1, kv=6000, kv_min=700, lens=5, Hq=32, Hkv=8,
             d=128, page=16, out="bf16"),
        # long ragged contexts with outlier key channels (the long-context configuration)
        _step("decode_long_16", B=16, kv=131072, kv_min=8192, lens=7, Hq=16, Hkv=8, outliers=True),
        # verification of 8-token draft chains at 16K keys (a published shape), K/V contiguous
        _step("verify_chain_8x16k", B=8, T=8, kv=16384, Hq=16, Hkv=8, page=0),
        # verification of 16-node draft trees after 8K keys, digit tiles kept across steps
        _step("verify_tree_8x8k", B=8, T=16, kv=8192, Hq=16, Hkv=8, page=0, tree=True, digits=True),
        # causal prefill of one 4096-token prompt
        _step("prefill_4096", B=1, T=4096, kv=4096, Hq=16, Hkv=8, page=0),
        # decode of a model with 64-dim heads
        _step("decode_d64_ragged", B=16, kv=8192, kv_min=1024, lens=9, Hq=32, Hkv=8, d=64),
        # causal prefill of a model with 64-dim heads
        _step("prefill_d64_2048", B=1, T=2048, kv=2048, Hq=32, Hkv=8, d=64, page=0),
        # a mixed serving batch: one prompt chunk among decoding sequences
        dict(name="forward_mixed_12", kind="forward", B=12, tok=1, last=150, kv=5000, kv_min=300, lens=11, Hq=16,
             Hkv=8, d=128, page=16, out="bf16"),
        # one head's causal rows on host arrays, fp32 result (the fixture's shape)
        dict(name="host_causal_2048", kind="host", rows=2048, d=128, out="fp32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: no more keys read or pairs scored than the largest listed."""
    kind = rng.choice(["decode", "decode", "decode", "verify", "verify", "prefill", "prefill", "forward", "hf", "host"])
    Hkv = rng.choice([4, 8])
    grp = rng.choice([1, 2, 4, 8])
    d = rng.choice([128, 128, 128, 64, 96])
    page = rng.choice([0, 16, 16, 64])
    out = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    lens = rng.randrange(1 << 20)
    if kind == "decode":
        B = _log(rng, 1, 48)
        kv = _log(rng, 100, min(131072, 400_000 // B))
        return _step(None, B=B, kv=kv, kv_min=rng.choice([kv, max(1, kv // 8)]), lens=lens, Hq=Hkv * grp, Hkv=Hkv, d=d,
                     page=page, out=out, outliers=rng.random() < 0.25)
    if kind == "verify":
        # draft trees keep their digit tiles (128-dim heads) about half the time
        T, B = _log(rng, 2, 24), _log(rng, 1, 16)
        kv = _log(rng, max(T, 200), min(32768, 400_000 // (B * grp) + T))
        tree = rng.random() < 0.5
        return _step(None, B=B, T=T, kv=kv, kv_min=rng.choice([kv, max(T, kv // 4)]), lens=lens, Hq=Hkv * grp, Hkv=Hkv,
                     d=d, page=page, out=out, tree=tree, digits=d == 128 and rng.random() < 0.4)
    if kind == "prefill":
        # at most the pairs of the listed prefill of that head width
        lim = 4096 * 4096 * 8 if d == 128 else 2048 * 2048 * 16
        T = _log(rng, 24, 3000)
        kv = min(T + rng.choice([0, 0, _log(rng, 50, 6000)]), max(T, lim // (T * Hkv * grp)))
        if T * kv * Hkv * grp > lim:
            T = kv = int(math.sqrt(lim / (Hkv * grp)))
        return _step(None, B=1, T=T, kv=kv, Hq=Hkv * grp, Hkv=Hkv, d=d, page=page, out=out)
    if kind == "forward":
        B = _log(rng, 2, 32)
        shape = rng.choice(["decode", "verify", "mixed"])
        tok = rng.randint(2, 8) if shape == "verify" else 1
        last = _log(rng, 16, 300) if shape == "mixed" else tok
        return dict(kind="forward", B=B, tok=tok, last=last, kv=_log(rng, 400, 8000), kv_min=100, lens=lens, Hq=Hkv * min(grp, 4),
                    Hkv=Hkv, d=rng.choice([128, 128, 64]), page=rng.choice([16, 64]), out=out)
    if kind == "hf":
        kl = _log(rng, 40, 6000)
        return dict(kind="hf", B=_log(rng, 1, 4), ql=rng.choice([1, 1, min(kl, _log(rng, 2, 200))]), kl=kl, Hq=Hkv * grp,
                    Hkv=Hkv, d=d)
    return dict(kind="host", rows=_log(rng, 60, 2048), d=d, out=rng.choice(["bf16", "fp32"]))


# ---- what a case holds

def _lens(case):
    """Key counts of the case's sequences (without a tree's nodes)."""
    lo, hi, B = case["kv_min"], case["kv"], case["B"]
    if lo == hi:
        return [hi] * B
    r = random.Random(case["lens"])
    return [hi] + [_log(r, lo, hi) for _ in range(B - 1)]


def _ql(case):
    """New tokens per sequence of a "forward" case."""
    return [case["tok"]] * (case["B"] - 1) + [case["last"]]


def _normal(shape, gen):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(generator=gen)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


class _State:
    pass


def _step_inputs(case, seed):
    """The step's tensors and its problem dict (exactattention_amd.problem's keys)."""
    gen, r = _gen(seed), np.random.default_rng(seed)
    B, T, Hq, Hkv, d = case["B"], case["T"], case["Hq"], case["Hkv"], case["d"]
    tree = case["tree"]
    lens = _lens(case)
    total = [n + (T if tree else 0) for n in lens]
    S = max(total)
    q = _normal((B, T, Hq, d), gen)
    P = case["page"]
    if P:
        npp = -(-S // P)
        need = [-(-n // P) for n in total]
        perm = r.permutation(sum(need)).astype(np.int32)
        bt, at = np.zeros((B, npp), np.int32), 0
        for b, n in enumerate(need):
            bt[b, :n] = perm[at:at + n]
            at += n
        shape, strides = (sum(need), P, Hkv, d), (P * Hkv * d, Hkv * d, d)
        hdim = 2
    else:
        bt = None
        shape, strides = (B, Hkv, S, d), (Hkv * S * d, d, S * d)
        hdim = 1
    k, v = _normal(shape, gen), _normal(shape, gen)
    if case["outliers"]:
        scale = torch.ones((Hkv, d), device="cuda", dtype=torch.bfloat16)
        for h in range(Hkv):
            scale[h, torch.from_numpy(r.choice(d, size=4, replace=False)).cuda()] = 30.0
        k *= scale if hdim == 2 else scale[:, None, :]
    mask = base = None
    if tree:
        kv_len = np.repeat(np.asarray(lens, np.int32)[:, None], T, 1)
        mask = np.zeros((B, T), np.uint64)
        for b in range(B):
            parent = configs.draft_tree(r, T, 6)
            for i in range(T):
                m = 0
                for a in configs.path_of(parent, i):
                    m |= 1 << a
                mask[b, i] = m
        base = np.asarray(lens, np.int32)
    else:
        kv_len = np.asarray(lens, np.int32)[:, None] - T + 1 + np.arange(T, dtype=np.int32)
    geom = dict(num_seqs=B, num_tokens=T, num_q_heads=Hq, num_kv_heads=Hkv, head_dim=d, head_dim_v=d,
                q_seq_stride=T * Hq * d, q_tok_stride=Hq * d, q_head_stride=d, o_seq_stride=T * Hq * d,
                o_tok_stride=Hq * d, o_head_stride=d, k_page_stride=strides[0], k_slot_stride=strides[1],
                k_head_stride=strides[2], v_page_stride=strides[0], v_slot_stride=strides[1],
                v_head_stride=strides[2], page_size=P or 1, block_table_stride=0 if bt is None else bt.shape[1],
                max_seq_len=S)
    return dict(geom=geom, q=q, k=k, v=v, seq_len=np.asarray(total, np.int32),
                kv_len=np.ascontiguousarray(kv_len).reshape(-1), block_table=bt,
                tree_mask=None if mask is None else mask.reshape(-1), tree_base=base, out_shape=(B, T, Hq, d))


def _bf16_host(rows, d, gen):
    return _normal((rows, d), gen).view(torch.int16).cpu().numpy().view(np.uint16)


def _forward_inputs(case, seed):
    gen = _gen(seed)
    lens, n = _lens(case), sum(_ql(case))
    Hq, Hkv, d = case["Hq"], case["Hkv"], case["d"]
    prefix = [(_normal((m, Hkv, d), gen), _normal((m, Hkv, d), gen)) for m in lens]
    return lens, prefix, _normal((n, Hq, d), gen), _normal((n, Hkv, d), gen), _normal((n, Hkv, d), gen)


def _hf_inputs(case, seed):
    gen = _gen(seed)
    B, d = case["B"], case["d"]
    return (_normal((B, case["Hq"], case["ql"], d), gen), _normal((B, case["Hkv"], case["kl"], d), gen),
            _normal((B, case["Hkv"], case["kl"], d), gen))


def _host_inputs(case, seed):
    gen = _gen(seed)
    return tuple(_bf16_host(case["rows"], case["d"], gen) for _ in range(3))


def prepare(case, seed):
    s = _State()
    s.kind, s.d = case["kind"], case["d"]
    if s.kind == "step":
        s.dp = hip.DeviceProblem(_step_inputs(case, seed), case["out"])
        s.alpha = default_alpha_bits(case["d"])
        s.dig = None
        if case["digits"]:
            S = s.dp.geom["max_seq_len"]
            s.dig = hip.KVDigits(s.dp, -(-S // 64))
            s.dig.update(s.dp, torch.zeros_like(s.dp.t["seq_len"]), s.dp.t["seq_len"], S)
    elif s.kind == "forward":
        s.lens, prefix, s.q, s.k, s.v = _forward_inputs(case, seed)
        P, extra = case["page"], max(_ql(case))
        pages = sum(-(-(n + extra) // P) for n in s.lens)
        s.cache = PagedKVCache(pages, P, case["Hkv"], case["d"], case["B"], max(s.lens) + extra)
        s.be = ExactAttentionBackend(s.cache, case["Hq"], out=case["out"], alpha_bits=default_alpha_bits(case["d"]))
        s.seqs = [s.cache.add_sequence() for _ in s.lens]
        for i, (pk, pv) in zip(s.seqs, prefix):
            s.cache.append(i, pk, pv)
        s.ql = _ql(case)
    elif s.kind == "hf":
        s.q, s.k, s.v = _hf_inputs(case, seed)
        s.scaling = case["d"] ** -0.5
    else:
        s.q, s.k, s.v = _host_inputs(case, seed)
        s.kv_len = np.arange(1, case["rows"] + 1)
        s.alpha, s.out = ea.default_alpha(case["d"]), case["out"]
    return s


def run(s):
    if s.kind == "step":
        hip.launch_hip(s.dp, s.alpha, kv_digits=s.dig)
        return s.dp.out.view(torch.float32 if s.dp.out_fp32 else torch.bfloat16), s.dp.flags
    if s.kind == "forward":
        for i, n in zip(s.seqs, s.lens):
            s.cache.truncate(i, n)
        out, flags = s.be.forward(s.q, s.k, s.v, s.seqs, s.ql)
        return out.view(torch.float32 if s.be.out == "fp32" else torch.bfloat16), flags
    if s.kind == "hf":
        return hf_attention(None, s.q, s.k, s.v, scaling=s.scaling)[0]
    return ea.attention_hip(s.q, s.k, s.v, s.alpha, kv_len=s.kv_len, out=s.out)


# ---- what a pass cannot do without

def work(case):
    """K and V read once, q read and the output written once; 2 d flops per scored pair for q.k
    and as many for P.V."""
    d = case["d"]
    if case["kind"] == "step":
        B, T, Hq, Hkv = case["B"], case["T"], case["Hq"], case["Hkv"]
        lens = _lens(case)
        keys = sum(lens) + (B * T if case["tree"] else 0)
        # a tree node sees the prefix and about 3 nodes of its path
        pairs = sum(T * n + 3 * T for n in lens) if case["tree"] else sum(T * n - T * (T - 1) // 2 for n in lens)
        rows, osz = B * T * Hq, 4 if case["out"] == "fp32" else 2
    elif case["kind"] == "forward":
        Hq, Hkv = case["Hq"], case["Hkv"]
        lens = _lens(case)
        # the new keys are read, written and attended
        keys = sum(lens) + 3 * sum(_ql(case))
        pairs = sum(q * n + q * (q + 1) // 2 for q, n in zip(_ql(case), lens))
        rows, osz = sum(_ql(case)) * Hq, 4 if case["out"] == "fp32" else 2
    elif case["kind"] == "hf":
        B, ql, kl, Hq, Hkv = case["B"], case["ql"], case["kl"], case["Hq"], case["Hkv"]
        keys, pairs, rows, osz = B * kl, B * (ql * kl - ql * (ql - 1) // 2), B * ql * Hq, 2
    else:
        n = case["rows"]
        Hq = Hkv = 1
        keys, pairs, rows, osz = n, n * (n + 1) // 2, n, 4 if case["out"] == "fp32" else 2
    return {"bytes": keys * Hkv * 4 * d + rows * d * (2 + osz), "flops": pairs * Hq * 4 * d}


def tolerance(case):
    return "exact"


# ---- the same attention in 64 bits

def _attend(q, k, v, alpha, kvl, extra=None):
    """q (T, Hq, d), k/v (n, Hkv, d) -> (T, Hq, d) float64; token t sees keys below kvl[t], plus
    the keys of extra[t] (a boolean (T, n) mask)."""
    T, Hq, d = q.shape
    n, Hkv = k.shape[0], k.shape[1]
    grp = Hq // Hkv
    out = torch.empty((T, Hq, d), dtype=torch.float64, device=q.device)
    pos = torch.arange(n, device=q.device)
    vis = pos[None, :] < kvl[:, None]
    if extra is not None:
        vis = vis | extra
    step = max(1, 64_000_000 // max(n * grp, 1))  # tokens at a time: bounds the score matrix
    for h in range(Hkv):
        kh, vh = k[:, h].double().contiguous(), v[:, h].double().contiguous()
        for t0 in range(0, T, step):
            t1 = min(T, t0 + step)
            qh = q[t0:t1, h * grp:(h + 1) * grp].double().reshape(-1, d)
            s = (qh @ kh.t().contiguous()) * alpha
            m = vis[t0:t1].repeat_interleave(grp, 0)
            s = torch.where(m, s, torch.full_like(s, -math.inf))
            w = torch.exp2(s - s.amax(1, keepdim=True))
            out[t0:t1, h * grp:(h + 1) * grp] = ((w @ vh) / w.sum(1, keepdim=True)).view(t1 - t0, grp, d)
    return out


def exact(case, seed):
    d = case["d"]
    if case["kind"] == "step":
        p = _step_inputs(case, seed)
        g = p["geom"]
        alpha = float(np.uint32(default_alpha_bits(d)).view(np.float32))
        B, T = case["B"], case["T"]
        out = torch.empty(p["out_shape"], dtype=torch.float64, device="cuda")
        kvl = torch.from_numpy(p["kv_len"]).cuda().view(B, T)
        for b in range(B):
            n = int(p["seq_len"][b])
            if p["block_table"] is not None:
                idx = torch.from_numpy(p["block_table"][b][:-(-n // g["page_size"])]).cuda().long()
                kb, vb = (p[x][idx].reshape(-1, case["Hkv"], d)[:n] for x in ("k", "v"))
            else:
                kb, vb = (p[x][b, :, :n].transpose(0, 1) for x in ("k", "v"))
            extra = None
            if p["tree_mask"] is not None:
                e = np.zeros((T, n), bool)
                L = int(p["tree_base"][b])
                for t in range(T):
                    m = int(p["tree_mask"][b * T + t])
                    e[t, L:L + T] = [(m >> i) & 1 for i in range(T)]
                extra = torch.from_numpy(e).cuda()
            out[b] = _attend(p["q"][b], kb, vb, alpha, kvl[b], extra)
        return out, None
    if case["kind"] == "forward":
        lens, prefix, q, k, v = _forward_inputs(case, seed)
        alpha = float(np.uint32(default_alpha_bits(d)).view(np.float32))
        out, at = [], 0
        for n, ql, (pk, pv) in zip(lens, _ql(case), prefix):
            kvl = n + 1 + torch.arange(ql, device="cuda")
            out.append(_attend(q[at:at + ql], torch.cat([pk, k[at:at + ql]]), torch.cat([pv, v[at:at + ql]]), alpha, kvl))
            at += ql
        return torch.cat(out), None
    if case["kind"] == "hf":
        q, k, v = _hf_inputs(case, seed)
        kl, ql = case["kl"], case["ql"]
        alpha = float(np.float32(d ** -0.5 / math.log(2)))
        kvl = kl - ql + 1 + torch.arange(ql, device="cuda")
        return torch.stack([_attend(q[b].transpose(0, 1), k[b].transpose(0, 1), v[b].transpose(0, 1), alpha, kvl)
                            for b in range(case["B"])])
    if case["out"] == "bf16":
        return None  # bit patterns, not numbers
    q, k, v = (torch.from_numpy(x.view(np.int16)).cuda().view(torch.bfloat16)[:, None] for x in _host_inputs(case, seed))
    kvl = 1 + torch.arange(case["rows"], device="cuda")
    out = _attend(q, k, v, float(np.float32(ea.default_alpha(d))), kvl)
    return out[:, 0].cpu().numpy(), None
