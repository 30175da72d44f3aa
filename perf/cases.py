"""The calls that programs make of this framework, for timing and comparing.

``listed()`` names them, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass
through the public entry points of ``moonmath_attention``, and ``exact`` is
what the pass computes, in 64 bits.

Kinds of cases:

* ``attn``   -- ``forward``: self- and cross-attention of diffusion transformers
  and their text encoders (bf16 in, bf16 out).
* ``lite``   -- ``forward_lite``: one denoising step over a skip list.
* ``mla``    -- the absorbed-MLA decode ops over an fp8 cache: contiguous slabs,
  flat-slot pages and 64-token block tables, one query or a draft window.
* ``kv``     -- ``mla_kv_quantize``: new tokens written into the fp8 cache.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "amd-kernels_amd"))

import moonmath_attention as ma  # noqa: E402

DEV = "cuda:0"
D, LAT, ROPE, QK, PAGE = 128, 512, 64, 576, 64
KV_SCALE = 1.0 / 32.0
MLA_SCALE = 1.0 / math.sqrt(192.0)  # qk head dim 128 + 64
LITE_THRESHOLD = -6.0               # the LiteAttention class's default
QROWS, KROWS, WAVE_ROWS = 256, 64, 32  # a skip list's tile; rows that share a vote
MAX_FLOPS = 4.0 * 2 * 24 * 8192 * 8192 * D  # the largest listed case


def listed():
    return [
        # The smallest call: the README example's head count at 256 tokens.
        # Launches and host work are all there is to it.
        _attn("attn_tiny_2x256", 1, 2, 256, 256, "bhsd", "rtna", 1.0),
        # An image's tokens with a text prompt appended: ragged in both
        # directions and fewer q-blocks than the chip has CUs.
        _attn("attn_image_24x1531", 1, 24, 1531, 1531, "bshd", "rtna", 1.0),
        # The benchmark's video-length self-attention.
        _attn("attn_video_48x8192", 2, 24, 8192, 8192, "bshd", "rtne", 1.0),
        # Cross-attention of that video to a 77-token prompt and to a 512-token
        # one (an odd number of query rows).
        _attn("attn_cross_8192x77", 2, 24, 8192, 77, "bshd", "rtne", 0.5),
        _attn("attn_cross_4097x512", 2, 24, 4097, 512, "bshd", "rtna", 0.5),
        # A later denoising step: the skip lists keep about a quarter.
        {"name": "lite_video_keep25", "kind": "lite", "B": 2, "H": 24, "S": 8192, "keep": 0.25, "layout": "bshd",
         "mode": "rtna"},
        # Serving, 64 requests of 1K..8K tokens: one rank of eight (16 heads),
        # and all 128 heads on one GPU.
        _mla("mla_b64_h16", 64, 16, 1, 1024, 8192, "flat"),
        _mla("mla_b64_h128", 64, 128, 1, 1024, 8192, "flat"),
        # Speculative decoding: windows of 4 drafts on one rank of eight, and
        # of 2 with all heads over block tables.
        _mla("mla_draft4_b32_h16", 32, 16, 4, 1024, 8192, "flat"),
        _mla("mla_draft2_b64_h128", 64, 128, 2, 1024, 8192, "blocks"),
        # One conversation on its own: latency of a single 4097-token request.
        _mla("mla_b1_h16_4097", 1, 16, 1, 4097, 4097, "slab"),
        # A prompt's tokens entering the cache.
        {"name": "kv_write_8192", "kind": "kv", "N": 8192, "saturate": False},
    ]


def _attn(name, B, H, Sq, Skv, layout, mode, k_gain):
    return {"name": name, "kind": "attn", "B": B, "H": H, "Sq": Sq, "Skv": Skv, "layout": layout, "mode": mode,
            "k_gain": k_gain}


def _mla(name, B, H, q_len, lo, hi, cache):
    return {"name": name, "kind": "mla", "B": B, "H": H, "q_len": q_len, "lo": lo, "hi": hi, "cache": cache}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "cross", "cross", "lite", "mla", "mla", "mla", "mla", "kv"])
    if kind in ("attn", "cross"):
        while True:
            B, H = rng.choice([1, 1, 2, 4]), rng.choice([2, 3, 8, 12, 16, 24, 32])
            Sq = _log_int(rng, 64, 16384)
            # Self-attention, or a longer / shorter set of keys.
            Skv = _log_int(rng, 16, 1024) if kind == "cross" else (Sq if rng.random() < 0.75 else _log_int(rng, 64, 16384))
            if 4.0 * B * H * Sq * Skv * D <= MAX_FLOPS and B * H * (Sq + Skv) <= 1 << 20:
                break
        c = _attn("", B, H, Sq, Skv, rng.choice(["bhsd", "bshd"]), rng.choice(["rtna", "rtne", "rtz"]),
                  0.5 if kind == "cross" else 1.0)
    elif kind == "lite":
        c = {"name": "", "kind": "lite", "B": rng.choice([1, 2]), "H": rng.choice([2, 8, 16, 24]),
             "S": _log_int(rng, 1024, 8192), "keep": rng.choice([0.15, 0.25, 0.5, 1.0]),
             "layout": rng.choice(["bhsd", "bshd"]), "mode": rng.choice(["rtna", "rtne"])}
    elif kind == "mla":
        while True:
            B, H, q_len = _log_int(rng, 1, 128), rng.choice([8, 16, 16, 32, 64, 128]), rng.choice([1, 1, 1, 2, 3, 4, 8])
            lo = _log_int(rng, 128, 8192)
            hi = lo if rng.random() < 0.3 else _log_int(rng, lo, 16384)
            if B * hi <= 64 * 8192 and B * hi * H * q_len <= 64 * 8192 * 256:
                break
        c = _mla("", B, H, q_len, lo, hi, rng.choice(["flat", "flat", "blocks", "slab"]))
    else:
        c = {"name": "", "kind": "kv", "N": _log_int(rng, 16, 65536), "saturate": rng.random() < 0.5}
    del c["name"]
    return c


# ---- inputs ------------------------------------------------------------------------------


def _rand(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _qkv(case, g, Sq, Skv):
    """N(0, 1) activations; key norms are log-normal around that (a few keys
    draw most of the attention) times ``k_gain``."""
    B, H = case["B"], case["H"]
    shape = (lambda s: (B, H, s, D)) if case["layout"] == "bhsd" else (lambda s: (B, s, H, D))
    q, k, v = _rand(g, *shape(Sq)), _rand(g, *shape(Skv)), _rand(g, *shape(Skv))
    gain = case.get("k_gain", 1.0)
    k = k * (torch.exp(0.25 * _rand(g, *k.shape[:3], 1)) * gain)
    if gain != 1.0:
        v = v * gain
    return q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)


def _lens(case, g):
    if case["lo"] == case["hi"] or case["cache"] == "slab":
        return [case["hi"]] * case["B"]
    return torch.randint(case["lo"], case["hi"] + 1, (case["B"],), generator=g, device=DEV).tolist()


def _fp8_rows(g, n):
    """Cache rows as ``mla_kv_quantize`` leaves them: N(0, 1) codes."""
    return torch.randn(n, QK, generator=g, device=DEV).to(torch.float8_e4m3fn)


def _skip_rows(case, g, nqb, nkb):
    """[B*H*nqb, nkb] bool: the kept blocks; the first one always."""
    keep = torch.rand(case["B"] * case["H"] * nqb, nkb, generator=g, device=DEV) < case["keep"]
    keep[:, 0] = True
    return keep


def _skip_list(keep):
    """Kept blocks as run-length rows walked in ascending order: [len, e1 - 1,
    s1 - 1, ...], the runs [s, e) from the last to the first."""
    n, nkb = keep.shape
    k = torch.cat([torch.zeros(n, 1, dtype=torch.bool, device=DEV), keep,
                   torch.zeros(n, 1, dtype=torch.bool, device=DEV)], 1)
    edge = k[:, 1:] != k[:, :-1]                       # position b: the state changes at block b
    rows = torch.zeros(n, nkb + 2, dtype=torch.int16, device=DEV)
    count = edge.sum(1)
    rows[:, 0] = count.to(torch.int16)
    after = edge.flip(1).cumsum(1).flip(1)              # 1-based place from the end
    r, b = torch.nonzero(edge, as_tuple=True)
    rows[r, after[r, b]] = (b - 1).to(torch.int16)
    return rows


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = case["kind"]
    if kind == "attn":
        q, k, v = _qkv(case, g, case["Sq"], case["Skv"])
        return {"kind": kind, "q": q, "k": k, "v": v, "mode": case["mode"], "layout": case["layout"]}
    if kind == "lite":
        q, k, v = _qkv(case, g, case["S"], case["S"])
        B, H, nqb, nkb = case["B"], case["H"], -(-case["S"] // QROWS), -(-case["S"] // KROWS)
        read = _skip_list(_skip_rows(case, g, nqb, nkb)).view(B, H, nqb, nkb + 2)
        return {"kind": kind, "q": q, "k": k, "v": v, "read": read, "write": torch.zeros_like(read),
                "mode": case["mode"], "layout": case["layout"]}
    if kind == "mla":
        B, H, n = case["B"], case["H"], case["q_len"]
        lens = _lens(case, g)
        # The draft window is a dimension of its own where there is one.
        lead = (B, H) if n == 1 else (B, n, H)
        s = {"kind": kind, "cache": case["cache"], "multi": n > 1, "q_lat": _rand(g, *lead, LAT).to(torch.bfloat16),
             "q_pe": _rand(g, *lead, ROPE).to(torch.bfloat16),
             "o": torch.zeros(*lead, LAT, dtype=torch.bfloat16, device=DEV)}
        if case["cache"] == "slab":
            s["kv"] = _fp8_rows(g, B * lens[0]).view(B, lens[0], QK)
            return s
        pages = [-(-x // PAGE) for x in lens]
        pool_pages = int(math.ceil(sum(pages) * 1.25))
        order = torch.randperm(pool_pages, generator=g, device=DEV).to(torch.int32)
        s["kv"] = _fp8_rows(g, pool_pages * PAGE).view(pool_pages, PAGE, QK)
        s["lens"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        plan = ma.mla_decode_a16w8_multiq_plan_parts_q if n > 1 else ma.mla_decode_a16w8_plan_parts_q
        s["parts"] = plan(B, case["hi"], n, H)
        if case["cache"] == "blocks":
            table = torch.zeros(B, max(pages), dtype=torch.int32, device=DEV)
            at = 0
            for b, p in enumerate(pages):
                table[b, :p] = order[at:at + p]
                at += p
            s["table"] = table
            return s
        s["kv"] = s["kv"].view(pool_pages * PAGE, 1, QK)
        idx, at = [], 0
        for x, p in zip(lens, pages):
            slots = order[at:at + p].view(p, 1) * PAGE + torch.arange(PAGE, dtype=torch.int32, device=DEV)
            idx.append(slots.view(-1)[:x])
            at += p
        s["indices"] = torch.cat(idx)
        s["indptr"] = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
        return s
    N = case["N"]
    slots_n = N + N // 4 + PAGE
    return {"kind": "kv", "c_kv": (_rand(g, N, LAT) * KV_SCALE).to(torch.bfloat16),
            "k_pe": (_rand(g, N, ROPE) * KV_SCALE).to(torch.bfloat16), "saturate": case["saturate"],
            "pool": torch.zeros(slots_n, 1, QK, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn),
            "slots": torch.randperm(slots_n, generator=g, device=DEV)[:N].to(torch.int32)}


# ---- one pass ----------------------------------------------------------------------------


def run(s):
    kind = s["kind"]
    if kind == "attn":
        return ma.forward(s["q"], s["k"], s["v"], round_mode=s["mode"], layout=s["layout"])
    if kind == "lite":
        out = ma.forward_lite(s["q"], s["k"], s["v"], s["read"], s["write"], threshold=LITE_THRESHOLD, phase=1,
                              round_mode=s["mode"], layout=s["layout"])
        return out, s["write"]
    if kind == "mla":
        if s["cache"] == "slab":
            op = ma.mla_decode_a16w8_multiq if s["multi"] else ma.mla_decode_a16w8
            op(s["q_lat"], s["q_pe"], s["kv"], s["o"], MLA_SCALE, KV_SCALE)
        elif s["cache"] == "blocks":
            ma.mla_decode_a16w8_paged_blocks(s["q_lat"], s["q_pe"], s["kv"], s["o"], s["lens"], s["table"],
                                             s["parts"], MLA_SCALE, KV_SCALE)
        else:
            op = ma.mla_decode_a16w8_multiq_paged_dev if s["multi"] else ma.mla_decode_a16w8_paged_dev
            op(s["q_lat"], s["q_pe"], s["kv"], s["o"], s["lens"], None, s["indices"], s["indptr"], s["parts"],
               MLA_SCALE, KV_SCALE)
        return s["o"]
    ma.mla_kv_quantize(s["c_kv"], s["k_pe"], s["pool"], s["slots"], KV_SCALE, s["saturate"])
    return s["pool"].view(torch.uint8)


# ---- what a pass cannot do without -------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "attn":
        bh, Sq, Skv = case["B"] * case["H"], case["Sq"], case["Skv"]
        return {"bytes": 4.0 * bh * D * (Sq + Skv), "flops": 4.0 * bh * Sq * Skv * D}
    if kind == "lite":
        bh, S = case["B"] * case["H"], case["S"]
        lists = 2.0 * 2 * bh * -(-S // QROWS) * (-(-S // KROWS) + 2)
        kept = min(1.0, case["keep"] + (1.0 - case["keep"]) / -(-S // KROWS))  # the first block always
        return {"bytes": 8.0 * bh * D * S + lists, "flops": 4.0 * bh * S * S * D * kept}
    if kind == "mla":
        one = case["lo"] == case["hi"] or case["cache"] == "slab"
        tokens = case["B"] * (case["hi"] if one else (case["lo"] + case["hi"]) / 2)
        rows = case["B"] * case["H"] * case["q_len"]
        index = {"slab": 0, "flat": 4, "blocks": 4 / PAGE}[case["cache"]] * tokens
        return {"bytes": tokens * QK + index + rows * (QK + LAT) * 2.0,
                "flops": 2.0 * (QK + LAT) * case["H"] * case["q_len"] * tokens}
    return {"bytes": case["N"] * (2.0 * QK + QK + 4), "flops": 0.0}


def tolerance(case):
    if case["kind"] == "kv":
        return "exact"  # bytes
    # bf16 results (half a unit in the last place: 2^-9, 1.7e-3 in the 2-norm)
    # of weights rounded to bf16 once more.
    t = {"rel": 8e-3, "max": 0.06}
    if case["kind"] == "lite":
        # A wave of 32 rows takes or drops a block by comparing fp32 scores;
        # a last bit can move a marker of the next list.
        t["differ"] = 1e-4
    return t


# ---- in 64 bits --------------------------------------------------------------------------


def _attend(q, k, v, scale):
    """softmax(q k^T scale) v of one head in 64 bits, by rows."""
    out = []
    for r in range(0, q.shape[0], 4096):
        p = torch.softmax(q[r:r + 4096] @ k.T * scale, -1)
        out.append(p @ v)
    return torch.cat(out)


def _attend_listed(q, k, v, scale, keep):
    """One head over the kept blocks of each 256-row tile, in ascending order. A
    wave of 32 rows takes a block for its rows when some row's best score comes
    within the threshold (log2) of that row's best over the blocks it took
    before; the first one always."""
    S, nkb = q.shape[0], keep.shape[1]
    out = torch.empty_like(q)
    c = scale * math.log2(math.e)
    for t in range(keep.shape[0]):
        rows = q[t * QROWS:(t + 1) * QROWS]
        s = rows @ k.T * c
        n = rows.shape[0]
        waves = -(-n // WAVE_ROWS)
        pad = torch.full((waves * WAVE_ROWS, nkb * KROWS), -math.inf, dtype=torch.float64, device=q.device)
        pad[:n, :S] = s
        best = pad.view(waves, WAVE_ROWS, nkb, KROWS).amax(-1)
        blocks = torch.nonzero(keep[t]).flatten().tolist()
        took = torch.zeros(waves, nkb, dtype=torch.bool, device=q.device)
        top = torch.full((waves, WAVE_ROWS), -math.inf, dtype=torch.float64, device=q.device)
        for i, b in enumerate(blocks):
            now = best[:, :, b]
            yes = (now > top + LITE_THRESHOLD).any(1) if i else torch.ones(waves, dtype=torch.bool, device=q.device)
            took[:, b] = yes
            top = torch.where(yes[:, None], torch.maximum(top, now), top)
        mask = took.repeat_interleave(WAVE_ROWS, 0)[:n].repeat_interleave(KROWS, 1)[:, :S]
        p = torch.softmax(s.masked_fill(~mask, -math.inf) * math.log(2.0), -1)
        out[t * QROWS:(t + 1) * QROWS] = p @ v
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "kv":
        return None  # bytes, compared as they are
    s = prepare(case, seed)
    if kind in ("attn", "lite"):
        heads = (lambda t: t) if case["layout"] == "bhsd" else (lambda t: t.transpose(1, 2))
        q, k, v = heads(s["q"]), heads(s["k"]), heads(s["v"])
        if kind == "lite":
            # Tiles times listed blocks, a few small steps each.
            nqb, nkb = -(-case["S"] // QROWS), -(-case["S"] // KROWS)
            if case["B"] * case["H"] * nqb * (1 + nkb * case["keep"]) > 1 << 16:
                return None
            g = torch.Generator(device=DEV).manual_seed(int(seed))
            _qkv(case, g, case["S"], case["S"])
            keep = _skip_rows(case, g, nqb, nkb).view(case["B"], case["H"], nqb, nkb)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                a = [t[b, h].double() for t in (q, k, v)]
                out[b, h] = (_attend(*a, 1.0 / math.sqrt(D)) if kind == "attn" else
                             _attend_listed(*a, 1.0 / math.sqrt(D), keep[b, h]))
        out = out if case["layout"] == "bhsd" else out.transpose(1, 2).contiguous()
        return out if kind == "attn" else (out, None)
    B, H, n = case["B"], case["H"], case["q_len"]
    ql = s["q_lat"].view(B, n * H, LAT).double()
    qp = s["q_pe"].view(B, n * H, ROPE).double()
    out = torch.empty(B, n * H, LAT, dtype=torch.float64, device=DEV)
    lens = s["lens"].tolist() if "lens" in s else [s["kv"].shape[1]] * B
    at = 0
    for b, L in enumerate(lens):
        if s["cache"] == "slab":
            rows = s["kv"][b]
        elif s["cache"] == "blocks":
            rows = s["kv"].view(torch.uint8)[s["table"][b, :-(-L // PAGE)].long()].view(-1, QK)[:L].view(torch.float8_e4m3fn)
        else:
            rows = s["kv"].view(torch.uint8).view(-1, QK)[s["indices"][at:at + L].long()].view(torch.float8_e4m3fn)
            at += L
        kv = rows.to(torch.float32).double() * KV_SCALE
        sc = (ql[b] @ kv[:, :LAT].T + qp[b] @ kv[:, LAT:].T) * MLA_SCALE
        # Draft position t sees all but the last n - 1 - t tokens.
        seen = L - (n - 1) + torch.arange(n, device=DEV).repeat_interleave(H)
        sc = sc.masked_fill(torch.arange(L, device=DEV)[None] >= seen[:, None], -math.inf)
        out[b] = torch.softmax(sc, -1) @ kv[:, :LAT]
    return out.view(s["o"].shape)
