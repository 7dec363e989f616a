"""The calls a user of this package makes, as timed cases over the range of sizes it is used at.

Every case is a dict of plain values with a "kind":

  flat     fast_article_causal_attention (block coresets, compressor "sorted_pair")
  exact    fast_article_causal_attention with compressor "none" (exact attention)
  levels   article_causal_attention (merge-and-reduce levels)
  segment  triton_article_causal_attention (segment-mean coresets)
  flash    triton_flash_causal_attention (exact softmax attention)
  decode   ArticleStreamingAttention after a prefix: one pass is one block of tokens, token by token
  prompt   a new ArticleStreamingAttention taking a prompt: prefill() outputs and the state it leaves

`exact` states each of them in plain float64 torch: the Taylor part from Kronecker powers of the keys, the
residual over the coreset items that the seeded draws select, the exact in-block part.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("streaming-attention_amd"))

import fast_article_attention as fast  # noqa: E402
import streaming_taylor_coreset_attention as streaming  # noqa: E402
import triton_article_attention as gpu_api  # noqa: E402

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def listed():
    return [
        # one short sequence at the command line's default sizes (the smallest call: launches and latency)
        dict(name="flat_1x1024_d32", kind="flat", batch=0, heads=1, n=1024, d=32, dv=32, dtype="float32", degree=2,
             block=128, scale=1.0, data="ball", radius=1.0),
        # batched prefill of ordinary 64-wide heads with 16-bit inputs
        dict(name="flat_8x16x4096_bf16", kind="flat", batch=8, heads=16, n=4096, d=64, dv=64, dtype="bfloat16",
             degree=2, block=256, scale=0.125, data="normal", radius=1.0),
        # the long-context prefill that the benchmark quotes
        dict(name="levels_32x65536", kind="levels", batch=1, heads=32, n=65536, d=64, dv=64, dtype="float32",
             degree=2, block=256, scale=0.125, data="ball", radius=1.0),
        # the higher-degree configuration: narrow keys, 969 features, logits up to 2.25
        dict(name="levels_4x32x16384_deg3", kind="levels", batch=4, heads=32, n=16384, d=16, dv=64, dtype="float32",
             degree=3, block=128, scale=1.0, data="ball", radius=1.5),
        # a few heads of one long document: ragged length, widths that are no power of two
        dict(name="levels_3x12345_d40_f16", kind="levels", batch=1, heads=3, n=12345, d=40, dv=72, dtype="float16",
             degree=2, block=192, scale=None, data="ball", radius=1.0),
        # the exact option of the fast path on a batch of medium sequences
        dict(name="exact_4x8x2048", kind="exact", batch=4, heads=8, n=2048, d=64, dv=64, dtype="float32", degree=2,
             block=128, scale=0.125, data="ball", radius=1.0),
        # the segment-mean API with its command line's half-precision inputs, ragged length
        dict(name="segment_2x8x3000_f16", kind="segment", batch=2, heads=8, n=3000, d=64, dv=64, dtype="float16",
             degree=2, block=128, stride=2, scale=None, data="ball", radius=1.0),
        # the exact baseline, 16-bit inputs (what a user compares the approximation against)
        dict(name="flash_2x16x8192_bf16", kind="flash", batch=2, heads=16, n=8192, d=64, dv=64, dtype="bfloat16",
             scale=None, data="normal", radius=1.0),
        # the exact baseline, float32, odd length
        dict(name="flash_8x8191_f32", kind="flash", batch=1, heads=8, n=8191, d=64, dv=64, dtype="float32",
             scale=None, data="ball", radius=1.0),
        # serving: 64 sequences x 32 heads decoding in lockstep, one block completion in each pass
        dict(name="decode_2048_streams_bf16", kind="decode", streams=2048, prefix=8192, d=64, dv=64,
             dtype="bfloat16", degree=2, block=256, scale=0.125, data="normal", radius=0.125, fused=True),
        # one sequence through the reference's own update() and query(), token by token
        dict(name="decode_1_stream", kind="decode", streams=0, prefix=1000, d=64, dv=64, dtype="float32", degree=2,
             block=128, scale=None, data="ball", radius=1.0, fused=False),
        # a new session: 2 sequences x 32 heads take a 2000-token prompt, outputs and state
        dict(name="prompt_64x2000_bf16", kind="prompt", streams=64, n=2000, d=64, dv=64, dtype="bfloat16", degree=2,
             block=256, scale=0.125, data="normal", radius=0.5),
    ]


def _between(rng, lo, hi):
    """A whole number in [lo, hi], uniform over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["flat", "levels", "levels", "exact", "segment", "flash", "flash", "decode", "prompt"])
    d = rng.choice([16, 32, 40, 64, 64, 64, 80, 96, 128])
    dv = rng.choice([d, d, 16, 32, 64, 72, 128])
    dtype = rng.choice(["float32", "bfloat16", "float16"])
    scale = None if rng.random() < 0.7 else round(rng.uniform(0.05, 1.0), 3)
    degree = rng.choice([1, 2, 2, 2])
    block = rng.choice([64, 100, 128, 128, 192, 256, 256, 512])
    common = dict(kind=kind, d=d, dv=dv, dtype=dtype, scale=scale, data="ball", radius=1.0)
    if kind == "flash":
        n = _between(rng, 200, 16384)
        heads = _between(rng, 1, max(1, min(64, (64 * 8192 * 8192) // (n * n * max(d, dv)))) if dtype == "float32"
                         else max(1, min(128, (64 * 32 * 8192 * 8192) // (n * n * max(d, dv)))))
        return dict(common, batch=1, heads=heads, n=n)
    if kind == "exact":
        n = _between(rng, 200, 4096)
        return dict(common, batch=1, heads=_between(rng, 1, max(1, min(64, 64 * 32 * 2048 * 2048 // (n * n * d)))),
                    n=n, degree=degree, block=block)
    if kind == "segment":
        n = _between(rng, 200, 8192)
        return dict(common, batch=1, heads=_between(rng, 1, min(64, 1 + 262144 // n)), n=n, degree=degree, block=block,
                    stride=rng.choice([s for s in (2, 4, 8) if block % s == 0]))
    if kind == "flat":
        n = _between(rng, 200, 8192)
        return dict(common, batch=1, heads=_between(rng, 1, max(1, min(128, 64 * 262144 // (n * d)))), n=n,
                    degree=degree, block=block)
    if kind == "levels":
        if d <= 16:
            degree = rng.choice([2, 3])
        n = _between(rng, 300, 65536)
        return dict(common, batch=1, heads=_between(rng, 1, max(1, min(64, 64 * 524288 // (n * d)))), n=n,
                    degree=degree, block=block)
    d = min(d, 64)
    dv = min(dv, 64)
    if kind == "prompt":
        n = _between(rng, 200, 6000)
        return dict(common, d=d, dv=dv, streams=_between(rng, 1, min(128, 1 + 262144 // n)), n=n, degree=degree,
                    block=block)
    streams = _between(rng, 1, 512)
    return dict(common, d=d, dv=dv, streams=streams, prefix=_between(rng, 100, 4096), degree=degree, block=block,
                fused=rng.random() < 0.7)


# ------------------------------------------------------------------------------------------- inputs


def _rows(g, lead, width, case, value=False):
    x = torch.randn(*lead, width, device="cuda", generator=g)
    if not value and case["data"] == "ball":  # uniform in the ball of the radius
        r = torch.rand(*lead, 1, device="cuda", generator=g).pow_(1.0 / width) * case["radius"]
        x = x / torch.linalg.vector_norm(x, dim=-1, keepdim=True).clamp_(min=1e-12) * r
    elif case["data"] == "normal":
        x *= case["radius"]
    return x.to(DTYPES[case["dtype"]])


def _qkv(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    if case["kind"] == "prompt":
        lead = (case["streams"], case["n"])
    elif case["batch"] == 0:
        lead = (case["n"],)
    else:
        lead = (case["batch"], case["heads"], case["n"])
    q = _rows(g, lead, case["d"], case)
    k = _rows(g, lead, case["d"], case)
    return q, k, _rows(g, lead, case["dv"], case, value=True)


def _decode_inputs(case, seed):
    """The prefix's keys and values [S, P, .] and the next block's tokens [T, S, .]."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    s, t = max(1, case["streams"]), case["block"]
    k = _rows(g, (s, case["prefix"]), case["d"], case)
    v = _rows(g, (s, case["prefix"]), case["dv"], case, value=True)
    tok = (_rows(g, (t, s), case["d"], case), _rows(g, (t, s), case["d"], case),
           _rows(g, (t, s), case["dv"], case, value=True))
    return k, v, tok


def _session(case):
    return streaming.ArticleStreamingAttention(case["d"], case["dv"], degree=case["degree"], block_size=case["block"],
                                               scale=case["scale"], dtype=DTYPES[case["dtype"]],
                                               streams=case["streams"] or None)


def prepare(case, seed):
    if case["kind"] == "decode":
        k, v, (tq, tk, tv) = _decode_inputs(case, seed)
        att = _session(case)
        one = case["streams"] == 0
        att.extend(k[0] if one else k, v[0] if one else v)
        if one:
            tq, tk, tv = tq[:, 0].contiguous(), tk[:, 0].contiguous(), tv[:, 0].contiguous()
        return {"case": case, "att": att, "q": tq, "k": tk, "v": tv}
    q, k, v = _qkv(case, seed)
    return {"case": case, "q": q, "k": k, "v": v}


# --------------------------------------------------------------------------------------------- one pass


def run(state):
    c, q, k, v = state["case"], state["q"], state["k"], state["v"]
    kind = c["kind"]
    if kind == "flat" or kind == "exact":
        return fast.fast_article_causal_attention(q, k, v, degree=c["degree"], block_size=c["block"],
                                                  scale=c["scale"],
                                                  compressor="none" if kind == "exact" else "sorted_pair")
    if kind == "levels":
        return streaming.article_causal_attention(q, k, v, degree=c["degree"], block_size=c["block"],
                                                  scale=c["scale"])
    if kind == "segment":
        return gpu_api.triton_article_causal_attention(q, k, v, degree=c["degree"], block_size=c["block"],
                                                       compress_stride=c["stride"], scale=c["scale"])
    if kind == "flash":
        return gpu_api.triton_flash_causal_attention(q, k, v, scale=c["scale"])
    if kind == "prompt":
        att = _session(c)
        out = att.prefill(q, k, v)
        return {"out": out, "num": att.sketch.num_moments, "den": att.sketch.den_moments,
                "levels": [None if b is None else (b.keys, b.values, b.weights) for b in att.coreset.levels]}
    att, outs = state["att"], []
    for t in range(q.shape[0]):
        if c["fused"]:
            outs.append(att.step(q[t], k[t], v[t]))
        else:
            att.update(k[t], v[t])
            outs.append(att.query(q[t]))
    return torch.stack(outs)


# --------------------------------------------------------------------------- what a pass cannot do without


def _per_row(case, n, first=0):
    """Coreset items that a row reads on average, over the rows [first, n)."""
    b = case["block"]
    m = (b + 1) // 2
    if case["kind"] in ("flat", "segment"):
        m = m if case["kind"] == "flat" else b // case["stride"]
        return m * (n / b - 1) / 2 if n > b else 0.0
    c0, c1 = first // b, max(n // b, first // b + 1)
    return m * sum(bin(c).count("1") for c in range(c0, c1)) / (c1 - c0)


def work(case):
    kind, d, dv = case["kind"], case["d"], case["dv"]
    es = 4 if case["dtype"] == "float32" else 2
    pair = 2 * d + 2 * (dv + 1)
    if kind == "flash" or kind == "exact":
        rows = max(1, case["batch"]) * case["heads"] * case["n"]
        out = 4 if kind == "flash" else es
        return {"bytes": rows * ((2 * d + dv) * es + dv * out), "flops": rows * (case["n"] + 1) / 2 * pair}
    feats = math.comb(d + case["degree"], case["degree"])
    if kind == "decode":
        s, t = max(1, case["streams"]), case["block"]
        items = _per_row(case, case["prefix"] + t, case["prefix"])
        state = feats * (dv + 1) * 4
        token = state + items * (d + dv + 1) * 4 + t / 2 * (d + dv) * 4 + (2 * d + 2 * dv) * es
        flops = 2 * feats * (dv + 1) + (items + t / 2) * pair
        return {"bytes": s * (t * token + 2 * state), "flops": s * t * (flops + 2 * feats * (dv + 1))}
    n = case["n"]
    rows = (case["streams"] if kind == "prompt" else max(1, case["batch"]) * case["heads"]) * n
    # the Taylor part by feature moments, or over the pairs where a sequence is too short for that
    low = min(4 * feats * (dv + 1), (n + 1) / 2 * pair)
    nbytes = rows * ((2 * d + dv) * es + dv * (4 if kind == "segment" else es))
    if kind == "prompt":
        nbytes += case["streams"] * (feats * (dv + 1) * 4 + _per_row(case, n, n) * (d + dv + 1) * 4)
    return {"bytes": nbytes, "flops": rows * (low + (_per_row(case, n) + min(case["block"], n) / 2) * pair)}


def tolerance(case):
    # measured against exact(): 1.3e-7 to 4.9e-6 where the outputs are float32 (products of operands carried in
    # two 16-bit halves, sums in another order), 1.7e-3 for bfloat16 and 1.9e-4 for float16 outputs (rounding)
    if case["kind"] in ("flash", "segment") or case["dtype"] == "float32":
        return {"rel": 2e-5}
    return {"rel": 8e-3} if case["dtype"] == "bfloat16" else {"rel": 1e-3}


# ------------------------------------------------------------------------------------- float64 statement


def _poly(x, degree):
    total, term = torch.ones_like(x), torch.ones_like(x)
    for r in range(1, degree + 1):
        term = term * x / r
        total = total + term
    return total


def _kron(x, r):
    out = torch.ones_like(x[..., :1])
    for _ in range(r):
        out = (out[..., :, None] * x[..., None, :]).flatten(-2)
    return out


def _low_sums(q, k, v1, degree, first=0, chunk=2048):
    """sum over j <= i of the Taylor polynomial of q_i.k_j times v1_j, for the rows [first, N) of [H, N, .]
    (q holds those rows only); the keys before a chunk through Kronecker moments."""
    h, n, d = k.shape
    group = max(1, (1 << 27) // (chunk * d ** degree))
    parts = []
    for h0 in range(0, h, group):
        qg, kg, vg = q[h0: h0 + group], k[h0: h0 + group], v1[h0: h0 + group]
        mom = [torch.zeros(kg.shape[0], d ** r, vg.shape[-1], device=k.device, dtype=k.dtype)
               for r in range(degree + 1)]
        rows = []
        edges = sorted(set(list(range(0, first, chunk)) + list(range(first, n, chunk)) + [n]))
        for lo, hi in zip(edges[:-1], edges[1:]):
            kc, vc = kg[:, lo:hi].contiguous(), vg[:, lo:hi].contiguous()
            if lo >= first:
                qc = qg[:, lo - first: hi - first].contiguous()
                x = torch.matmul(qc, kc.transpose(1, 2).contiguous())
                y = torch.matmul(_poly(x, degree).tril_(), vc)
                for r in range(degree + 1):
                    y += torch.matmul(_kron(qc, r), mom[r]) / math.factorial(r)
                rows.append(y)
            for r in range(degree + 1):
                mom[r] += torch.matmul(_kron(kc, r).transpose(1, 2).contiguous(), vc)
        parts.append(torch.cat(rows, 1))
    return torch.cat(parts)


class _Draws:
    """The compress calls' draws, one CPU generator for each sequence, in the order they are made."""

    def __init__(self, count, d):
        self.d, self.gens = d, []
        for s in range(count):
            g = torch.Generator()
            g.manual_seed(s)
            self.gens.append(g)

    def __call__(self, n):
        dirs, unif = [], []
        for g in self.gens:
            x = torch.randn(self.d, generator=g)
            dirs.append(x / torch.clamp(torch.linalg.vector_norm(x), min=1e-12))
            unif.append(torch.rand(n // 2, generator=g))
        return torch.stack(dirs).cuda().double(), torch.stack(unif).cuda()


def _take(x, idx):
    return x.gather(1, idx[..., None].expand(-1, -1, x.shape[-1]))


def _compress(k, src, w, draws):
    """One sorted_pair call for every sequence: neighbours of the projections' order, one of a pair kept."""
    n = src.shape[1]
    direction, u = draws(n)
    score = (_take(k, src) * direction[:, None, :]).sum(-1).float()
    order = torch.argsort(score, dim=1, stable=True)
    a, b = order[:, 0: n - n % 2: 2], order[:, 1: n: 2]
    wa, ws = w.gather(1, a), w.gather(1, a) + w.gather(1, b)
    keep = torch.where(u < wa / ws.clamp(min=1e-30), src.gather(1, a), src.gather(1, b))
    if n % 2:
        keep = torch.cat([keep, src.gather(1, order[:, -1:])], 1)
        ws = torch.cat([ws, w.gather(1, order[:, -1:])], 1)
    return keep, ws


def _block_node(k, j, block, draws):
    src = torch.arange(j * block, (j + 1) * block, device=k.device)[None].expand(k.shape[0], -1)
    return _compress(k, src, torch.ones(src.shape, device=k.device), draws)


def _level_sets(k, n, block):
    """The (src, w) lists of the levels after c completed blocks, c = 0, 1, ..., n // block."""
    draws = _Draws(k.shape[0], k.shape[-1])
    levels, sets = [], [[]]
    for c in range(n // block):
        cur, at = _block_node(k, c, block, draws), 0
        while at < len(levels) and levels[at] is not None:
            cur = _compress(k, torch.cat([levels[at][0], cur[0]], 1), torch.cat([levels[at][1], cur[1]], 1), draws)
            levels[at] = None
            at += 1
        levels += [None] * (at + 1 - len(levels))
        levels[at] = cur
        sets.append(list(levels))
    return sets


def _add_residual(sums, q, k, v1, degree, lo, hi, keys, first):
    """sums += exp minus its Taylor polynomial over the keys [keys, i] for the rows i of [lo, hi)."""
    qc = q[:, lo - first: hi - first].contiguous()
    x = torch.matmul(qc, k[:, keys:hi].transpose(1, 2).contiguous())
    late = torch.arange(keys, hi, device=k.device)[None, :] > torch.arange(lo, hi, device=k.device)[:, None]
    r = (torch.exp(x) - _poly(x, degree)).masked_fill_(late, 0.0)
    sums[:, lo - first: hi - first] += torch.matmul(r, v1[:, keys:hi].contiguous())


def _add_items(sums, q, degree, lo, hi, ik, iv1, w, first, clamp=None):
    qc = q[:, lo - first: hi - first].contiguous()
    x = torch.matmul(qc, ik.transpose(1, 2).contiguous())
    r = (torch.exp(x if clamp is None else x.clamp(max=clamp)) - _poly(x, degree)) * w[:, None, :]
    sums[:, lo - first: hi - first] += torch.matmul(r, iv1)


def _levels_exact(q, k, v1, case, sets, first=0):
    """The merge-and-reduce semantics for the rows [first, N)."""
    n, b, t = k.shape[1], case["block"], case["degree"]
    sums = _low_sums(q, k, v1, t, first)
    for c in range(n // b + 1):
        lo, hi = max(first, c * b - 1), min(n, (c + 1) * b - 1)
        if lo >= hi:
            continue
        if c * b < hi:  # the row that completes a block is answered from the levels alone
            _add_residual(sums, q, k, v1, t, lo, hi, c * b, first)
        nodes = [x for x in sets[c] if x is not None]
        if nodes:
            src, w = torch.cat([x[0] for x in nodes], 1), torch.cat([x[1] for x in nodes], 1).double()
            _add_items(sums, q, t, lo, hi, _take(k, src), _take(v1, src), w, first)
    return sums


def _divide(sums):
    return sums[..., :-1] / sums[..., -1:].clamp(min=1e-12)


def _with_ones(v):
    return torch.cat([v, torch.ones_like(v[..., :1])], -1)


def _softmax_rows(q, k, v1):
    h, n, d = k.shape
    out = torch.empty(h, n, v1.shape[-1] - 1, device=k.device, dtype=k.dtype)
    for i in range(h):
        for lo in range(0, n, 2048):
            hi = min(n, lo + 2048)
            x = q[i, lo:hi] @ k[i, :hi].t().contiguous()
            x += torch.full((hi - lo, hi), -math.inf, device=k.device, dtype=k.dtype).triu_(lo + 1)
            out[i, lo:hi] = torch.softmax(x, -1) @ v1[i, :hi, :-1]
    return out


def exact(case, seed):
    kind = case["kind"]
    s = 1.0 / math.sqrt(case["d"]) if case["scale"] is None else case["scale"]
    if kind == "decode":
        if max(1, case["streams"]) * (case["prefix"] // case["block"]) > 100_000:
            return None  # the draws alone take too long one call at a time
        k, v, (tq, tk, tv) = _decode_inputs(case, seed)
        k = torch.cat([k, tk.transpose(0, 1)], 1).double()
        v1 = _with_ones(torch.cat([v, tv.transpose(0, 1)], 1).double())
        q = tq.transpose(0, 1).double().contiguous() * s
        n, first, parts = k.shape[1], case["prefix"], []
        sets = _level_sets(k, n, case["block"])
        group = max(1, (1 << 27) // (n * (case["d"] + case["dv"])))
        for h in range(0, k.shape[0], group):
            cut = [[x if x is None else (x[0][h: h + group], x[1][h: h + group]) for x in c] for c in sets]
            parts.append(_divide(_levels_exact(q[h: h + group], k[h: h + group], v1[h: h + group], case, cut, first)))
        out = torch.cat(parts).transpose(0, 1)
        return out[:, 0] if case["streams"] == 0 else out
    q, k, v = _qkv(case, seed)
    lead = tuple(v.shape[:-1])
    flat = lambda x: x.reshape(-1, x.shape[-2], x.shape[-1]).double()  # noqa: E731
    q, k, v1 = flat(q) * s, flat(k), _with_ones(flat(v))
    if kind in ("flash", "exact"):
        return _softmax_rows(q, k, v1).reshape(*lead, -1)
    n, b, t = k.shape[1], case["block"], case["degree"]
    if kind in ("levels", "prompt"):
        sets = _level_sets(k, n, b)
        out = _divide(_levels_exact(q, k, v1, case, sets)).reshape(*lead, -1)
        if kind == "levels":
            return out
        return {"out": out, "num": _monomial_sums(k, v1[..., :-1], t), "den": [x[..., 0] for x in _monomial_sums(
            k, v1[..., -1:], t)], "levels": [None if x is None else (_take(k, x[0]), _take(v1, x[0])[..., :-1], x[1])
                                             for x in sets[-1]]}
    sums = _low_sums(q, k, v1, t)
    blocks = (n - 1) // b
    if kind == "flat":
        draws = _Draws(k.shape[0], k.shape[-1])
        nodes = [_block_node(k, j, b, draws) for j in range(blocks)]
        if nodes:
            src = torch.cat([x[0] for x in nodes], 1)
            ik, iv1, w = _take(k, src), _take(v1, src), torch.cat([x[1] for x in nodes], 1).double()
    else:
        st = case["stride"]
        ik, iv1 = (x[:, : blocks * b].reshape(x.shape[0], -1, st, x.shape[-1]).mean(2) for x in (k, v1))
        w = torch.full(ik.shape[:2], float(st), device=k.device, dtype=k.dtype)
    for j in range(blocks + 1):
        lo, hi = j * b, min(n, (j + 1) * b)
        _add_residual(sums, q, k, v1, t, lo, hi, lo, 0)
        if j:
            m = j * (w.shape[1] // blocks)
            _add_items(sums, q, t, lo, hi, ik[:, :m], iv1[:, :m].contiguous(), w[:, :m], 0,
                       80.0 if kind == "segment" else None)
    return _divide(sums).reshape(*lead, -1)


def _monomial_sums(k, v, degree):
    """Sums over the tokens of every monomial of the keys (non-decreasing index order) over its
    multiplicities' factorials, times the values: one tensor [H, F_r, dv] for each degree r."""
    out = []
    for r in range(degree + 1):
        idx = torch.combinations(torch.arange(k.shape[-1]), r, with_replacement=True) if r else torch.zeros(1, 0).long()
        coef = torch.ones(idx.shape[0], dtype=torch.float64)
        run_len = torch.ones(idx.shape[0], dtype=torch.float64)
        for p in range(1, r):
            run_len = torch.where(idx[:, p] == idx[:, p - 1], run_len + 1, torch.ones_like(run_len))
            coef /= run_len
        idx, coef = idx.to(k.device), coef.to(k.device)
        rows = []
        for h in range(k.shape[0]):
            f = torch.ones(k.shape[1], idx.shape[0], device=k.device, dtype=k.dtype)
            for p in range(r):
                f *= k[h][:, idx[:, p]]
            rows.append((f * coef).t().contiguous() @ v[h])
        out.append(torch.stack(rows))
    return out
