"""Performance cases of the compressed-domain attention path.

Each case is one call of a public entry point as a serving program makes it:
one layer's decode step, cache encode, prompt prefill or chunked prefill over a
paged cache of Hadamard-rotated codebook indices with per-token norms.

* ``listed()``   the named cases; ``draw(rng)`` one more of the same ranges.
* ``prepare``    inputs on the GPU, made from the seed alone.
* ``run``        one call; returns the tensors it wrote.
* ``work``       the bytes and operations the call cannot do without.
* ``exact``      the same quantity in float64 with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from sub0_amd.cda.kernels_cuda.fa2_cda import fa2_cda_prefill_varlen_v1
from sub0_amd.cda.kernels_cuda.wrappers import (
    decode_hmma_v1,
    hybrid_attn_v1,
    paged_encode_fused_cuda,
)

D = 128
DEV = "cuda:0"
KV_HEADS = 8          # heads of the benchmark configuration (32 query / 8 KV heads)


# ------------------------------------------------------------------ cases --

def _decode(lens_kind, B, N, H_kv=8, gs=4, levels=16, slot=0, block=16, two_cb=False):
    return dict(kind="decode", lens=lens_kind, B=B, N=N, H_kv=H_kv, gs=gs, levels=levels,
                slot=slot or (144 if levels == 16 else 80), block=block, two_cb=two_cb)


def _encode(T, H_kv=8, levels=16, slot=0):
    return dict(kind="encode", T=T, H_kv=H_kv, levels=levels,
                slot=slot or (144 if levels == 16 else 80))


def _prefill(kind, B, q_lo, q_hi, past, H_kv=8, gs=4, block=16):
    """B sequences of q_lo..q_hi new tokens, each after up to `past` cached ones."""
    return dict(kind=kind, B=B, q_lo=q_lo, q_hi=q_hi, past=past, H_kv=H_kv, gs=gs, block=block)


def listed():
    named = {
        # One user generating with a short context: the latency of a token.
        "decode_b1_n4k": _decode("full", 1, 4096),
        # A small batch of requests of different lengths, K and V with a
        # trained codebook each (the two codebook arguments of the call).
        "decode_b4_ragged_two_codebooks": _decode("ragged", 4, 16001, two_cb=True),
        # The benchmark's headline: a full batch over long contexts.
        "decode_b32_n64k": _decode("full", 32, 65536),
        # 2-bit codes, the smaller cache format.
        "decode_k2v2_b32_n16k": _decode("full", 32, 16384, levels=4),
        # One rank of four that share 64 query / 8 KV heads by tensor
        # parallelism: two KV heads with eight queries each.
        "decode_tp4_gqa8_b16_n16k": _decode("ragged", 16, 16384, H_kv=2, gs=8),
        # A serving engine that sizes its pages for fp16 K and V (the memory
        # saving left off): 512-byte slots that hold the same codes.
        "decode_slot512_b8_n8k": _decode("full", 8, 8192, slot=512),
        # The cache update of one decode step.
        "encode_step_b32": _encode(32),
        # The cache update of a batch of prompts (64 sequences, ragged).
        "encode_prompt_8002": _encode(8002),
        # Eight prompts of 512..8192 tokens.
        "prefill_batch8": _prefill("prefill", 8, 512, 8192, 0),
        # One prompt of ordinary length.
        "prefill_prompt_1987": _prefill("prefill", 1, 1987, 1987, 0),
        # Chunked prefill: 512-token chunks after 5K..8K cached tokens.
        "prefill_chunk512_past8k": _prefill("prefill", 4, 512, 512, 8192),
        # Chunked prefill whose chunk keeps its fresh fp16 K/V (merged with
        # the compressed prefix).
        "hybrid_b2_q300_past5k": _prefill("hybrid", 2, 200, 300, 5000),
    }
    return [dict(case, name=name) for name, case in named.items()]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "decode", "encode", "prefill", "chunk",
                       "hybrid"])
    heads = rng.choice([8, 8, 4, 2, 1])
    if kind == "decode":
        levels = rng.choice([16, 16, 4])
        slot = rng.choice([0, 0, 512]) if levels == 16 else 0
        # The wide slots move whole 64-byte segments: cap the largest cache.
        tokens = 32 * (8192 if slot else 65536)
        B = _log_int(rng, 1, 32)
        N = _log_int(rng, 64, min(65536, tokens // B))
        return _decode(rng.choice(["full", "ragged"]), B, N, heads, rng.choice([4, 4, 8]), levels,
                       slot, rng.choice([16, 16, 32]), rng.random() < 0.25)
    if kind == "encode":
        levels = rng.choice([16, 16, 4])
        return _encode(_log_int(rng, 1, 8192), heads, levels,
                       512 if levels == 16 and rng.random() < 0.3 else 0)
    if kind == "prefill":
        hi = _log_int(rng, 32, 8192)
        return _prefill("prefill", rng.randint(1, 8), max(1, hi // 16), hi, 0, heads,
                        rng.choice([4, 4, 8]) if heads < 8 else 4)
    hi = _log_int(rng, 16, 512)
    return _prefill("hybrid" if kind == "hybrid" else "prefill", rng.randint(1, 4),
                    max(1, hi // 2), hi, _log_int(rng, 64, 8192), heads,
                    rng.choice([4, 4, 8]) if heads < 8 else 4)


# ----------------------------------------------------------------- inputs --

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _codebook(levels, laplace=False):
    """Lloyd-Max centroids of the coordinates of a rotated unit vector in 128
    dimensions, taken as Gaussian (or, for a second table, as Laplacian)."""
    x = np.linspace(-0.5, 0.5, 20001)
    s = 1.0 / math.sqrt(D)
    w = np.exp(-np.abs(x) * math.sqrt(2.0) / s) if laplace else np.exp(-0.5 * (x / s) ** 2)
    c = np.quantile(np.repeat(x, np.maximum(1, (w * 50).astype(int))),
                    (np.arange(levels) + 0.5) / levels)
    for _ in range(200):
        i = np.searchsorted(0.5 * (c[1:] + c[:-1]), x)
        c = np.array([(w * x)[i == k].sum() / w[i == k].sum() for k in range(levels)])
    return torch.tensor(c, dtype=torch.float32, device=DEV)


_TABLES = {}


def _tables(case):
    """(cb_K, cb_V, R) as fp32 tensors on the GPU; cb_V is cb_K unless the case
    gives each its own."""
    key = (case.get("levels", 16), case.get("two_cb", False))
    if key not in _TABLES:
        cbk = _codebook(key[0])
        cbv = _codebook(key[0], laplace=True) if key[1] else cbk
        h = torch.ones(1, 1, dtype=torch.float64)
        while h.shape[0] < D:
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        _TABLES[key] = (cbk, cbv, (h / math.sqrt(D)).float().to(DEV))
    return _TABLES[key]


def _raw_k(g, *shape):
    """fp16 keys: N(0, 1) with four outlier channels eight times as large."""
    x = torch.randn(*shape, D, device=DEV, generator=g)
    x[..., [5, 37, 70, 101]] *= 8.0
    return x.half()


def _pack(codes, levels):
    """uint8 codes (..., 128) -> packed bytes, first dimension in the high bits."""
    if levels == 16:
        return (codes[..., 0::2] << 4) | codes[..., 1::2]
    return (codes[..., 0::4] << 6) | (codes[..., 1::4] << 4) | (codes[..., 2::4] << 2) \
        | codes[..., 3::4]


def _quantise(x, cb, R):
    y = (x.float() @ R).half().float()
    n = y.norm(dim=-1)
    mid = 0.5 * (cb[1:] + cb[:-1])
    return torch.bucketize(y / n.unsqueeze(-1), mid).to(torch.uint8), n


def _fill_cache(g, rows, H_kv, levels, slot, cbk, cbv, R):
    """A cache of `rows` slots holding encoded keys and values."""
    cache = torch.zeros(rows, H_kv, slot, dtype=torch.uint8, device=DEV)
    kb = D * (4 if levels == 16 else 2) // 8
    step = max(1, (1 << 18) // H_kv)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        ck, nk = _quantise(_raw_k(g, n, H_kv), cbk, R)
        cv, nv = _quantise(torch.randn(n, H_kv, D, device=DEV, generator=g).half(), cbv, R)
        dst = cache[r:r + n]
        dst[..., :kb] = _pack(ck, levels)
        dst[..., kb:2 * kb] = _pack(cv, levels)
        dst[..., 2 * kb:2 * kb + 8] = torch.stack([nk, nv], -1).contiguous().view(torch.uint8)
    return cache


def _ragged(which, B, lo, hi):
    """B lengths in lo..hi, the first of them hi; host integers that depend on
    the case alone, so that a case is the same work for every seed."""
    n = np.random.default_rng(which).integers(lo, hi + 1, B)
    n[0] = hi
    return [int(v) for v in n]


def _paged(case, lens, g):
    """(cache, block table) of a paged cache with the sequences' blocks permuted."""
    cbk, cbv, R = _tables(case)
    block = case["block"]
    width = (max(lens) + block - 1) // block
    blocks = len(lens) * width + 3
    cache = _fill_cache(g, blocks * block, case["H_kv"], case.get("levels", 16),
                        case.get("slot", 144), cbk, cbv, R)
    perm = torch.randperm(blocks, device=DEV, generator=g)[:len(lens) * width]
    return cache, perm.view(len(lens), width).to(torch.int32)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _lens(case):
    """(new tokens, total keys) of each sequence."""
    B = case["B"]
    if case["kind"] == "decode":
        return [1] * B, ([case["N"]] * B if case["lens"] == "full"
                         else _ragged(1, B, max(1, case["N"] // 4), case["N"]))
    q = _ragged(2, B, case["q_lo"], case["q_hi"])
    past = _ragged(3, B, case["past"] * 5 // 8, case["past"])
    return q, [a + b for a, b in zip(q, past)]


def prepare(case, seed):
    g = _gen(seed)
    cbk, cbv, R = _tables(case)
    H_kv = case["H_kv"]
    s = dict(case=case, cbk=cbk, cbv=cbv, R=R, R16=R.half())
    if case["kind"] == "encode":
        T = case["T"]
        s["k"] = _raw_k(g, T, H_kv)
        s["v"] = torch.randn(T, H_kv, D, device=DEV, generator=g).half()
        s["cache"] = torch.zeros(T + 16, H_kv, case["slot"], dtype=torch.uint8, device=DEV)
        s["slots"] = torch.randperm(T + 16, device=DEV, generator=g)[:T].to(torch.int32)
        return s
    H_q = H_kv * case["gs"]
    q_lens, lens = _lens(case)
    T = sum(q_lens)
    s["cache"], s["bt"] = _paged(case, lens, g)
    s["q"] = torch.randn(T, H_q, D, device=DEV, generator=g).half()
    if case["kind"] != "decode":
        s["k"] = _raw_k(g, T, H_kv)
        s["v"] = torch.randn(T, H_kv, D, device=DEV, generator=g).half()
        s["cu"] = _i32([0] + list(np.cumsum(q_lens)))
        s["max_q"] = max(q_lens)
    s["lens"] = _i32(lens)
    s["max_k"] = max(lens)
    s["out"] = torch.empty_like(s["q"])
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "encode":
        paged_encode_fused_cuda(s["k"], s["v"], s["slots"], s["cache"], cb_K=s["cbk"],
                                cb_V=s["cbv"])
        return s["cache"]
    if c["kind"] == "decode":
        decode_hmma_v1(s["q"], s["cache"], s["bt"], s["lens"], s["out"], cb_K=s["cbk"],
                       cb_V=s["cbv"], rotation_fp32=s["R"], rotation_fp16=s["R16"],
                       group_size=c["gs"], block_size=c["block"], max_seq_len=s["max_k"])
    elif c["kind"] == "prefill":
        fa2_cda_prefill_varlen_v1(s["q"], s["cache"], s["bt"], s["cu"], s["lens"], s["out"],
                                  cb_K=s["cbk"], cb_V=s["cbv"], rotation_fp32=s["R"],
                                  group_size=c["gs"], block_size=c["block"],
                                  max_query_len=s["max_q"], max_seq_len=s["max_k"],
                                  fuse_fa2_epilogue=True)
    else:
        hybrid_attn_v1(s["q"], s["k"], s["v"], s["out"], s["cache"], s["bt"],
                       cu_seqlens_q=s["cu"], seq_lens=s["lens"], cb_K=s["cbk"], cb_V=s["cbv"],
                       rotation_fp32=s["R"], rotation_fp16=s["R16"], group_size=c["gs"],
                       block_size=c["block"], max_seq_len=s["max_k"], max_query_len=s["max_q"])
    return s["out"]


# ------------------------------------------------------------------- work --

def work(case):
    H_kv = case["H_kv"]
    code = D * (4 if case.get("levels", 16) == 16 else 2) // 8
    slot = 2 * code + 8                              # codes and norms of one token and head
    if case["kind"] == "encode":
        T = case["T"]
        # The rotation's order is part of the format: 10923 fused multiply-adds
        # a vector when the columns' shared prefixes are summed once.
        return dict(bytes=T * H_kv * (4 * D + slot) + 4 * T, flops=2 * 10923 * 2 * T * H_kv)
    H_q = H_kv * case["gs"]
    q_lens, lens = _lens(case)
    pages = sum((n + case["block"] - 1) // case["block"] for n in lens)
    rows = sum(q_lens)
    pairs = sum(q * (n - q) + q * (q + 1) // 2 for q, n in zip(q_lens, lens))
    read = sum(lens) * H_kv * slot + 4 * pages + 4 * len(lens)
    if case["kind"] == "hybrid":                     # the chunk's keys are read as fp16
        read += sum(q_lens) * H_kv * (4 * D - slot)
    return dict(bytes=read + 2 * rows * H_q * D * 2, flops=4 * H_q * D * pairs)


def tolerance(case):
    if case["kind"] == "encode":
        return "exact"
    # fp16 rotated queries, decoded keys, softmax weights and rotated outputs
    # put a result 6e-4 to 1.2e-3 (1.7e-3 with 2-bit codes) from float64 in the
    # 2-norm, its worst value 4e-3 to 4e-2: about four times that.
    return {"rel": 5e-3 if case.get("levels", 16) == 16 else 7e-3, "max": 0.15}


# ------------------------------------------------------------------ exact --

def _dense(s, b, h, n):
    """K and V rows (n, 128) of head h of sequence b in float64."""
    c = s["case"]
    levels, block = c.get("levels", 16), c["block"]
    kb = D * (4 if levels == 16 else 2) // 8
    t = torch.arange(n, device=DEV)
    rows = s["bt"][b].long()[t // block] * block + t % block
    raw = s["cache"][rows, h]
    norms = raw[:, 2 * kb:2 * kb + 8].contiguous().view(torch.float32).double()

    def decode(x, cb):
        shifts = (4, 0) if levels == 16 else (6, 4, 2, 0)
        idx = torch.stack([(x >> sh) & (levels - 1) for sh in shifts], -1).flatten(-2)
        return cb.double()[idx.long()]

    return decode(raw[:, :kb], s["cbk"]) * norms[:, :1], \
        decode(raw[:, kb:2 * kb], s["cbv"]) * norms[:, 1:]


def exact(case, seed):
    if case["kind"] == "encode":
        return None                                  # bytes whose rounding the format fixes
    s = prepare(case, seed)
    gs, R = case["gs"], s["R"].double()
    q = s["q"].double() @ R
    out = torch.zeros_like(q)
    q_lens, lens = _lens(case)
    row = 0
    for b, (m, n) in enumerate(zip(q_lens, lens)):
        for h in range(case["H_kv"]):
            K, V = _dense(s, b, h, n)
            if case["kind"] == "hybrid":             # the chunk's own keys stay fp16
                K = torch.cat([K[:n - m], s["k"][row:row + m, h].double() @ R])
                V = torch.cat([V[:n - m], s["v"][row:row + m, h].double() @ R])
            for i0 in range(0, m, 2048):
                i1 = min(m, i0 + 2048)
                seen = n - m + i1                    # keys visible to the last of these rows
                ahead = torch.arange(seen, device=DEV)[None] > \
                    (torch.arange(i0, i1, device=DEV) + n - m)[:, None]
                for hq in range(h * gs, (h + 1) * gs):
                    p = q[row + i0:row + i1, hq] @ K[:seen].T / math.sqrt(D)
                    p = torch.softmax(p.masked_fill_(ahead, -math.inf), -1)
                    out[row + i0:row + i1, hq] = p @ V[:seen]
        row += m
    return out @ R.T
