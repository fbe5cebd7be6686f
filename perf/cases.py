"""What a serving program has this library do, as cases that can be timed.

The listed cases follow one attention layer of a long-context model through
its life: the prompt's prefill (selector and hybrid attention), the freeze of
its cache into the four decode segments, and decode steps, from one short
sequence to a full batch of long ones.  The head shapes are 32 query / 8 key
heads, 64 / 8 and 32 / 2, all of head dimension 128.

Inputs are Gaussian with per-(key head, channel) key offsets ~ N(0, 2); 5% of
the prefix keys lie along the group's mean query direction, three standard
deviations long: the vertical lines that the selector is there to find.
`draw` spreads cases of the same paths over prefixes of 512 to 32768 tokens,
batches of 1 to 32, every bit width, both 16-bit types and both orders of the
[batch, head, token] axes in memory.
"""

import math

import torch

import hyquant_amd as hq
from hyquant_amd.d_stage_kv_cache import DStageKVCache, DStageLayerCache
from hyquant_amd.patch import causal_attention

D = 128
RHO = 0.05                 # share of the prefix kept as vertical lines
LONGEST = 32768
MOST_TOKENS = 16 * 8 * LONGEST       # batch * key heads * prefix of the largest decode case
TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one user, short context: a decode step is launch latency and little else
        dict(name="decode_b1_1k", path="decode", batch=1, q_heads=32, kv_heads=8, prefix=1024, window=128, staging=37,
             k_bits=4, v_bits=4, dtype="bf16"),
        # one user, 8K context: the headline decode step
        dict(name="decode_b1_8k", path="decode", batch=1, q_heads=32, kv_heads=8, prefix=8192, window=128, staging=64,
             k_bits=4, v_bits=4, dtype="bf16"),
        # a full batch of the longest contexts: HBM bandwidth
        dict(name="decode_b16_32k", path="decode", batch=16, q_heads=32, kv_heads=8, prefix=32768, window=128, staging=64,
             k_bits=4, v_bits=4, dtype="bf16"),
        # 16 query heads on each of two key heads, odd prefix, an fp16 model with 2-bit values
        dict(name="decode_gqa16_b24_13k_k4v2", path="decode", batch=24, q_heads=32, kv_heads=2, prefix=13001, window=256,
             staging=101, k_bits=4, v_bits=2, dtype="fp16"),
        # continuous batching: sequences of 700 to 32000 tokens in one call
        dict(name="decode_ragged_b16", path="ragged", batch=16, q_heads=32, kv_heads=8, shortest=700, longest=32000,
             window=128, staging=64, k_bits=4, v_bits=4, dtype="bf16"),
        # a cache in the per-(group, channel) scale format, read as it is
        dict(name="decode_legacy_b16_30k", path="legacy", batch=16, q_heads=32, kv_heads=8, prefix=30011, window=128,
             staging=64, k_bits=4, v_bits=4, dtype="bf16"),
        # a short prompt of an fp16 model, projections still in [token, head] order
        dict(name="prefill_1500", path="prefill", variant="int8", batch=1, q_heads=32, kv_heads=8, prompt=1531, window=128,
             dtype="fp16", order="token"),
        # an 8K prompt, int8 QK and fp16 PV, as the patched model calls it
        dict(name="prefill_8k", path="prefill", variant="int8", batch=1, q_heads=32, kv_heads=8, prompt=8192, window=128,
             dtype="bf16", order="token"),
        # the longest prompt, fp8 PV
        dict(name="prefill_32k_fp8", path="prefill", variant="int8_fp8pv", batch=1, q_heads=32, kv_heads=8, prompt=32768,
             window=128, dtype="bf16", order="head"),
        # the selector alone over a whole batch of prompts
        dict(name="select_b32_16k", path="select", batch=32, q_heads=32, kv_heads=8, prompt=16384, window=256, dtype="bf16",
             order="head"),
        # prefill to decode: the cache of a few ragged-length prompts becomes its four segments
        dict(name="freeze_b4_12k", path="freeze", batch=4, q_heads=32, kv_heads=8, prompt=12345, window=256, k_bits=4,
             v_bits=4, dtype="bf16", order="token"),
        # a whole turn of one layer: prompt, freeze, 150 decode steps with their appends and one flush
        dict(name="turn_2k_150", path="turn", batch=1, q_heads=32, kv_heads=8, prompt=1900, steps=150, window=128, k_bits=4,
             v_bits=4, dtype="bf16", order="token"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["decode", "decode", "decode", "ragged", "legacy", "prefill", "prefill", "prefill", "select",
                       "freeze", "turn"])
    q_heads, kv_heads = rng.choice([(32, 8), (32, 8), (64, 8), (32, 2)])
    c = dict(path=path, q_heads=q_heads, kv_heads=kv_heads, window=rng.choice([128, 256]),
             dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if path in ("decode", "ragged", "legacy"):
        n = _log_int(rng, 1024, LONGEST)
        c.update(batch=_log_int(rng, 1, min(32, MOST_TOKENS // (kv_heads * n))), staging=rng.randint(1, 127))
        if path == "legacy":
            c.update(prefix=n, k_bits=rng.choice([4, 4, 2]), v_bits=rng.choice([4, 4, 2]), dtype="bf16")
            return c
        kb, vb = rng.choice([(4, 4), (4, 4), (4, 2), (2, 4), (8, 8)])
        c.update(k_bits=kb, v_bits=vb)
        if kb == 8:
            c["batch"] = max(1, c["batch"] // 2)
        if path == "decode":
            c.update(prefix=n)
        else:
            c.update(batch=max(2, c["batch"]), shortest=_log_int(rng, 600, n), longest=n)
            if c["batch"] * n * kv_heads > MOST_TOKENS:
                c["longest"] = n // 2
                c["shortest"] = min(c["shortest"], n // 2)
        return c
    c.update(order=rng.choice(["token", "token", "head"]))
    if path == "prefill":
        n = _log_int(rng, 512, 28000)           # the other variants take longer than the listed fp8 PV at 32K
        if q_heads == 64 and n > 14000:
            n //= 2
        most = 28000 * 28000 * 32 // (n * n * q_heads)
        c.update(variant=rng.choice(["int8", "int8", "int8_fp8pv", "fp8qk", "window", "causal"]),
                 batch=_log_int(rng, 1, max(1, min(8, most))), prompt=n)
    elif path in ("select", "freeze"):
        n = _log_int(rng, 1024, LONGEST)
        c.update(batch=_log_int(rng, 1, max(1, min(32, 32 * 8 * 16384 // (n * kv_heads * (1 if path == "select" else 4))))),
                 prompt=n)
        if path == "select":
            c["batch"] = max(1, c["batch"] * 32 // q_heads)
        else:
            c.update(k_bits=4, v_bits=rng.choice([4, 2]))
    else:
        c.update(batch=_log_int(rng, 1, 4), prompt=_log_int(rng, 600, 6000), steps=rng.randint(20, 160), k_bits=4,
                 v_bits=rng.choice([4, 2]))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _rows(c, g, n, offset=None):
    """[batch * key heads, n, D] rows of the case's type."""
    x = _randn(g, c["batch"] * c["kv_heads"], n, D)
    if offset is not None:
        x += offset.repeat(c["batch"], 1)[:, None, :]
    return x.to(TYPES[c["dtype"]])


def _lines(c, g, n, offset):
    """Vertical-line keys: the head's offset plus a common direction."""
    u = _randn(g, c["kv_heads"], D)
    x = 3.0 * math.sqrt(D) * u / u.norm(dim=-1, keepdim=True) + offset
    return x.repeat(c["batch"], 1)[:, None, :].expand(-1, n, -1).to(TYPES[c["dtype"]]).contiguous()


def _quantise(x, bits):
    """Per-token symmetric codes (packed, the first channel in the low bits) and fp16 scales."""
    top = 2 ** (bits - 1) - 1
    x = x.float()
    scale = (x.abs().amax(-1).clamp(min=1e-5) / top).half()
    code = torch.round(x / scale.float()[..., None]).clamp(-top - 1, top).to(torch.int8)
    return _pack(code, bits), scale


def _pack(code, bits):
    if bits == 8:
        return code
    per = 8 // bits
    code = (code & (2 ** bits - 1)).reshape(*code.shape[:-1], -1, per)
    out = code[..., 0].clone()
    for i in range(1, per):
        out |= code[..., i] << (bits * i)
    return out


def _codes(packed, bits):
    """The signed codes of packed rows, float64."""
    if bits == 8:
        return packed.double()
    u = packed.to(torch.int16) & 255
    parts = [(u >> (bits * i)) & (2 ** bits - 1) for i in range(8 // bits)]
    u = torch.stack(parts, -1).reshape(*packed.shape[:-1], D)
    return (u - 2 ** bits * (u >= 2 ** (bits - 1))).double()


def _legacy_quantise(x, bits):
    """Per-(128 tokens, channel) fp16 scales and offset codes, the first channel in the high bits."""
    bh, n, _ = x.shape
    groups = -(-n // 128)
    scale = torch.empty(bh, groups, D, dtype=torch.float16, device=x.device)
    packed = torch.empty(bh, n, D * bits // 8, dtype=torch.uint8, device=x.device)
    zero = 8.0 if bits == 4 else 1.5
    for h in range(0, bh, 8):
        y = torch.nn.functional.pad(x[h:h + 8].float(), (0, 0, 0, groups * 128 - n)).reshape(-1, groups, 128, D)
        s = (y.abs().amax(2) / (2 ** (bits - 1) - 0.5)).half()
        u = torch.round(y / s.float()[:, :, None].clamp(min=1e-7) + zero).clamp(0, 2 ** bits - 1).to(torch.uint8)
        u = u.reshape(-1, groups * 128, D // (8 // bits), 8 // bits)[:, :n]
        b = torch.zeros_like(u[..., 0])
        for i in range(8 // bits):
            b |= u[..., i] << (8 - bits * (i + 1))
        scale[h:h + 8], packed[h:h + 8] = s, b
    return packed, scale


def _legacy_values(packed, scale, bits):
    """float64 values of one head's legacy rows: packed [n, D * bits / 8], scale [groups, D]."""
    u = packed.to(torch.int16)
    parts = [(u >> (8 - bits * (i + 1))) & (2 ** bits - 1) for i in range(8 // bits)]
    u = torch.stack(parts, -1).reshape(packed.shape[0], D).double() - (8.0 if bits == 4 else 1.5)
    return u * scale.double().repeat_interleave(128, 0)[:packed.shape[0]]


def _top_k(n):
    return min(n, max(1, math.ceil(n * RHO))) if n > 0 else 0


def _segments(n, window):
    """(quantised, vertical-line, window) tokens of a prompt of n after the freeze."""
    w = min(window, n)
    t = _top_k(n - 2 * w) if n > 2 * w else 0
    return n - w - t, t, w


def _ragged_lengths(c):
    """Lengths spaced evenly over their logarithm, the same for every seed."""
    lo, hi, b = c["shortest"], c["longest"], c["batch"]
    return [int(round(lo * (hi / lo) ** (i / (b - 1)))) for i in range(b)]


def _ragged_segments(c):
    out = []
    for n in _ragged_lengths(c):
        nq, t, w = _segments(n, c["window"])
        out.append((nq, t + c["staging"] + w))
    return out


def _prompt(c, g):
    """q, k, v [batch, heads, prompt, D]: vertical lines planted in k, `order` of the axes in memory."""
    b, hq_, hk, n, w = c["batch"], c["q_heads"], c["kv_heads"], c["prompt"], c["window"]
    dt = TYPES[c["dtype"]]

    def heads(h, off=None):
        if c["order"] == "token":
            x = torch.randn(b, n, h, D, generator=g, device="cuda", dtype=dt).transpose(1, 2)
        else:
            x = torch.randn(b, h, n, D, generator=g, device="cuda", dtype=dt)
        return x if off is None else x.add_(off.to(dt)[:, None, :])

    off = math.sqrt(2.0) * _randn(g, hk, D)
    q, k, v = heads(hq_), heads(hk, off), heads(hk)
    lines = int(RHO * n)
    if n > w and lines:
        u = q[:, :, -w:].float().mean(2).reshape(b, hk, hq_ // hk, D).mean(2)
        u = off + 3.0 * math.sqrt(D) * u / u.norm(dim=-1, keepdim=True)
        at = torch.rand(b, hk, n - w, generator=g, device="cuda").argsort(-1)[..., :min(lines, n - w)]
        k.scatter_(2, at[..., None].expand(-1, -1, -1, D), u.to(dt)[:, :, None, :].expand(-1, -1, at.shape[-1], -1))
    return q, k, v


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def prepare(c, seed):
    g = _generator(seed)
    c = dict(c)
    path = c["path"]
    bh = c["batch"] * c["kv_heads"]
    dt = TYPES[c["dtype"]]
    s = dict(case=c, repeat=c["q_heads"] // c["kv_heads"])
    if path in ("decode", "legacy"):
        off = math.sqrt(2.0) * _randn(g, c["kv_heads"], D)
        if path == "decode":
            nq, t, w = _segments(c["prefix"], c["window"])
            (s["kp"], s["ks"]), (s["vp"], s["vs"]) = (_quantise(_rows(c, g, nq, off), c["k_bits"]),
                                                      _quantise(_rows(c, g, nq), c["v_bits"]))
            s["q"] = _randn(g, c["batch"] * c["q_heads"], D, dtype=dt)
        else:
            nq, t, w = c["prefix"], c["prefix"] // 20, c["window"]
            s["kp"], s["ks"] = _legacy_quantise(_rows(c, g, nq, off), c["k_bits"])
            s["vp"], s["vs"] = _legacy_quantise(_rows(c, g, nq), c["v_bits"])
            s["q"] = _randn(g, c["batch"], c["q_heads"], 1, D, dtype=dt)
        s["segments"] = [_lines(c, g, t, off), _rows(c, g, t)]
        for n in (c["staging"], w):
            s["segments"] += [_rows(c, g, n, off), _rows(c, g, n)]
    elif path == "ragged":
        off = math.sqrt(2.0) * _randn(g, c["kv_heads"], D)
        sizes = _ragged_segments(c)
        order = torch.randperm(c["batch"], generator=torch.Generator().manual_seed(seed)).tolist()
        sizes = [sizes[i] for i in order]
        nq, nb = max(a for a, _ in sizes), max(b for _, b in sizes)
        s["kp"], s["ks"] = _quantise(_rows(c, g, nq, off), c["k_bits"])
        s["vp"], s["vs"] = _quantise(_rows(c, g, nq), c["v_bits"])
        s["q"] = _randn(g, c["batch"] * c["q_heads"], D, dtype=dt)
        s["k"], s["v"] = _rows(c, g, nb, off), _rows(c, g, nb)
        lens = torch.tensor(sizes, dtype=torch.int32, device="cuda").repeat_interleave(c["kv_heads"], 0)
        s["lens_quant"], s["lens_bf16"] = lens[:, 0].contiguous(), lens[:, 1].contiguous()
    else:
        s["q"], s["k"], s["v"] = _prompt(c, g)
        if path == "freeze":       # the prompt's queries are gone by then, but for the cache's tail
            s["q"] = s["q"][:, :, -c["window"]:].clone()
        if path == "turn":
            b, hq_, hk, n = c["batch"], c["q_heads"], c["kv_heads"], c["steps"]
            s["steps"] = [(_randn(g, b, hq_, 1, D, dtype=dt), _randn(g, b, hk, 1, D, dtype=dt),
                           _randn(g, b, hk, 1, D, dtype=dt)) for _ in range(n)]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def _attend_prompt(c, s):
    q, k, v, w = s["q"], s["k"], s["v"], c["window"]
    variant = c.get("variant", "int8")
    if variant == "window":
        return hq.sage_unified_attention(q, k, v, window_size=w)
    if variant == "causal":
        return causal_attention(q, k, v)
    idx = hq.compute_vertical_indices(q, k, w, RHO, kv_repeat=s["repeat"])
    if variant == "fp8qk":
        return hq.sage_vertical_attention_v2_fp8(q, k, v, idx, window_size=w)
    return hq.sage_vertical_attention_v2(q, k, v, idx, window_size=w, pv_mode="fp8" if variant == "int8_fp8pv" else "fp16")


def _cache_tensors(layer):
    return dict(k_packed=layer.k_quant_packed, v_packed=layer.v_quant_packed, k_scale=layer.k_scale, v_scale=layer.v_scale,
                k_topk=layer.k_topk, v_topk=layer.v_topk, k_window=layer.k_window, v_window=layer.v_window,
                topk=layer.topk_indices)


def run(s):
    c = s["case"]
    path = c["path"]
    if path == "decode":
        return hq.fused_d_stage_decode(s["q"], s["kp"], s["vp"], s["ks"], s["vs"], *s["segments"], c["k_bits"], c["v_bits"],
                                       kv_repeat=s["repeat"])
    if path == "ragged":
        return hq.fused_d_stage_decode_batched(s["q"], s["kp"], s["vp"], s["ks"], s["vs"], s["k"], s["v"], s["lens_quant"],
                                               s["lens_bf16"], c["k_bits"], c["v_bits"], kv_repeat=s["repeat"])
    if path == "legacy":
        return hq.splitk_decode_attention_k4v4_mma(s["q"], s["kp"], s["vp"], s["ks"], s["vs"], *s["segments"],
                                                   kv_repeat=s["repeat"], k_bits=c["k_bits"], v_bits=c["v_bits"])
    if path == "prefill":
        return _attend_prompt(c, s)
    if path == "select":
        return hq.compute_vertical_indices(s["q"], s["k"], c["window"], RHO, kv_repeat=s["repeat"])
    if path == "freeze":
        layer = DStageLayerCache(0, c["k_bits"], c["v_bits"], window_size=c["window"], top_ratio=RHO)
        layer.update_prefill(s["k"], s["v"])
        layer.save_query_tail(s["q"])
        layer.freeze(kv_repeat=s["repeat"])
        return _cache_tensors(layer)
    cache = DStageKVCache(num_layers=1, k_bits=c["k_bits"], v_bits_fn=lambda i: c["v_bits"], window_size=c["window"],
                          top_ratio=RHO)
    layer = cache.get_layer(0)
    layer.save_query_tail(s["q"])
    cache.update(s["k"], s["v"], 0)
    prompt = _attend_prompt(c, s)
    layer.freeze(kv_repeat=s["repeat"])
    outs = []
    for q, k, v in s["steps"]:
        cache.update(k, v, 0)
        outs.append(layer.decode_attention(q, s["repeat"]))
    return dict(prompt=prompt, steps=torch.cat(outs, 2), **_cache_tensors(layer))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _decode_work(tokens, rows, c, heads_q):
    """`tokens` quantised and `rows` 16-bit tokens summed over the key heads."""
    per = 16 * (c["k_bits"] + c["v_bits"]) + 4
    repeat = c["q_heads"] // c["kv_heads"]
    return {"bytes": tokens * per + rows * 4 * D + heads_q * 4 * D, "flops": 4 * D * repeat * (tokens + rows)}


def _prefill_work(c):
    b, n = c["batch"], c["prompt"]
    return {"bytes": b * n * D * 2 * (2 * c["q_heads"] + 2 * c["kv_heads"]), "flops": 2 * b * c["q_heads"] * n * n * D}


def _select_work(c, heads_out, prefix):
    b, hk = c["batch"], c["kv_heads"]
    return {"bytes": b * (hk * prefix * 2 * D + c["q_heads"] * min(c["window"], c["prompt"]) * 2 * D + heads_out * _top_k(prefix) * 8),
            "flops": 2 * D * b * heads_out * prefix}


def _freeze_work(c):
    """The keys, the values and the query tail read once, the four segments and the indices written once."""
    n, w = c["prompt"], min(c["window"], c["prompt"])
    nq, t, _ = _segments(n, c["window"])
    bh = c["batch"] * c["kv_heads"]
    per = 16 * (c["k_bits"] + c["v_bits"]) + 4
    return {"bytes": bh * (n * 4 * D + nq * per + (t + w) * 4 * D + t * 8) + c["batch"] * c["q_heads"] * w * 2 * D,
            "flops": 2 * D * bh * max(0, n - 2 * w)}


def _add(*works):
    return {k: sum(w[k] for w in works) for k in ("bytes", "flops")}


def work(c):
    path = c["path"]
    bh, heads_q = c["batch"] * c["kv_heads"], c["batch"] * c["q_heads"]
    if path == "decode":
        nq, t, w = _segments(c["prefix"], c["window"])
        return _decode_work(bh * nq, bh * (t + w + c["staging"]), c, heads_q)
    if path == "legacy":
        return _decode_work(bh * c["prefix"], bh * (c["prefix"] // 20 + c["window"] + c["staging"]), c, heads_q)
    if path == "ragged":
        sizes = _ragged_segments(c)
        return _decode_work(c["kv_heads"] * sum(a for a, _ in sizes), c["kv_heads"] * sum(b for _, b in sizes), c, heads_q)
    if path == "prefill":
        if c["variant"] in ("window", "causal"):
            return _prefill_work(c)
        prefix = max(0, c["prompt"] - c["window"])        # the keys are read by the attention already
        return _add(_prefill_work(c), {"bytes": 0, "flops": 2 * D * heads_q * prefix})
    if path == "select":
        return _select_work(c, c["q_heads"], max(0, c["prompt"] - c["window"]))
    if path == "freeze":
        return _freeze_work(c)
    nq, t, w = _segments(c["prompt"], c["window"])
    step = []
    for i in range(1, c["steps"] + 1):
        done = i // 128 * 128
        step.append(_decode_work(bh * (nq + done), bh * (t + w + i - done), c, heads_q))
    return _add(_prefill_work(c), _freeze_work(c), *step)


def tolerance(c):
    path = c["path"]
    if path in ("select", "freeze"):
        return "exact"                # indices, codes, scales and copied rows
    if path == "prefill" and c["variant"] == "int8_fp8pv":
        return {"rel": 5e-2}          # P rounded to e4m3 (2^-4) against a running maximum that another tiling moves
    return {"rel": 1e-2}              # 16-bit outputs and operands


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------


def _softmax_rows(q, k, v):
    """One key head: q [r, D], k / v [n, D], float64."""
    return torch.softmax(q @ k.T * D ** -0.5, -1) @ v


def _causal(q, k, v):
    b, h, n, _ = q.shape
    repeat = h // k.shape[1]
    out = torch.empty(b, h, n, D, dtype=torch.float64, device=q.device)
    chunk = 2048
    for i in range(b):
        for j in range(k.shape[1]):
            kd, vd = k[i, j].double(), v[i, j].double()
            for a in range(0, n, chunk):
                e = min(n, a + chunk)
                above = torch.ones(e - a, e, dtype=torch.bool, device=q.device).triu(a + 1)
                for m in range(repeat):
                    x = q[i, j * repeat + m, a:e].double() @ kd[:e].T
                    x = torch.softmax(x.mul_(D ** -0.5).masked_fill_(above, -math.inf), -1)
                    out[i, j * repeat + m, a:e] = x @ vd[:e]
    return out


def _exact_turn(c, s):
    """The decode steps over the cache as the freeze and the flush leave it."""
    b, hk, r, n, w = c["batch"], c["kv_heads"], s["repeat"], c["prompt"], min(c["window"], c["prompt"])
    dt = TYPES[c["dtype"]]
    p = max(0, n - 2 * w)
    t = _top_k(p)
    out = torch.empty(b, c["q_heads"], c["steps"], D, dtype=torch.float64, device="cuda")
    mean = s["q"][:, :, -w:].reshape(b, hk, r, w, D).double().mean(2).to(dt).double().mean(2).to(dt)
    for i in range(b):
        for j in range(hk):
            k, v = s["k"][i, j], s["v"][i, j]
            score = (k[:p].double() @ mean[i, j].double()).to(dt)
            top = torch.sort(score, descending=True, stable=True)[1][:t]
            rest = torch.ones(n - w, dtype=torch.bool, device="cuda")
            rest[top] = False

            def values(x, bits):
                packed, scale = _quantise(x, bits)
                return _codes(packed, bits) * scale.double()[:, None]

            kk = [values(k[:n - w][rest], c["k_bits"]), k[top].double(), k[n - w:].double()]
            vv = [values(v[:n - w][rest], c["v_bits"]), v[top].double(), v[n - w:].double()]
            new_k = torch.stack([x[1][i, j, 0] for x in s["steps"]])
            new_v = torch.stack([x[2][i, j, 0] for x in s["steps"]])
            kd, vd = values(new_k, c["k_bits"]), values(new_v, c["v_bits"])
            for m in range(c["steps"]):
                done = (m + 1) // 128 * 128
                keys = torch.cat(kk + [kd[:done], new_k[done:m + 1].double()])
                vals = torch.cat(vv + [vd[:done], new_v[done:m + 1].double()])
                q = s["steps"][m][0][i, j * r:(j + 1) * r, 0].double()
                out[i, j * r:(j + 1) * r, m] = _softmax_rows(q, keys, vals)
    return out


def exact(c, seed):
    path = c["path"]
    if path in ("select", "freeze"):
        return None                   # whole numbers and copies
    s = prepare(c, seed)
    r = s["repeat"]
    if path == "prefill":
        return _causal(s["q"], s["k"], s["v"])
    if path == "turn":
        none = dict.fromkeys(("k_packed", "v_packed", "k_scale", "v_scale", "k_topk", "v_topk", "k_window", "v_window", "topk"))
        return dict(prompt=_causal(s["q"], s["k"], s["v"]), steps=_exact_turn(c, s), **none)
    q = s["q"].reshape(-1, D).double()
    out = torch.empty_like(q)
    for h in range(c["batch"] * c["kv_heads"]):
        if path == "legacy":
            k = _legacy_values(s["kp"][h], s["ks"][h], c["k_bits"])
            v = _legacy_values(s["vp"][h], s["vs"][h], c["v_bits"])
        else:
            k = _codes(s["kp"][h], c["k_bits"]) * s["ks"][h].double()[:, None]
            v = _codes(s["vp"][h], c["v_bits"]) * s["vs"][h].double()[:, None]
        if path == "ragged":
            a, e = int(s["lens_quant"][h]), int(s["lens_bf16"][h])
            k, v = torch.cat([k[:a], s["k"][h, :e].double()]), torch.cat([v[:a], s["v"][h, :e].double()])
        else:
            seg = s["segments"]
            k = torch.cat([k] + [x[h].double() for x in seg[0::2]])
            v = torch.cat([v] + [x[h].double() for x in seg[1::2]])
        out[h * r:(h + 1) * r] = _softmax_rows(q[h * r:(h + 1) * r], k, v)
    return out.reshape(s["q"].shape)
