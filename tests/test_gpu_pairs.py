"""The pair kernel (sta_flash_attention_split, sta_exact_attention_split, sta_pair_moments) at the edges of its
tiles, key batches and tile orders, against float64 attention.  fp32 operands as three bf16 planes keep each product within 2^-23 of its
value and the sums are fp32: a few 2^-23 in the 2-norm (1e-6).  bf16 weights as hi + lo planes of 8 bits are
within 2^-16 each, uniform and of random sign (4e-6 at most in the 2-norm).  16-bit outputs add their rounding:
half a unit in the last of 8 (bf16) or 11 (fp16) bits at most, uniform, so 2^-8 / sqrt(3) or 2^-11 / sqrt(3)."""

import pytest
import torch

import _engine
import _native
import fast_article_attention as faa
import streaming_taylor_coreset_attention as stc
import triton_article_attention as taa

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = {torch.float32: 0.0, torch.bfloat16: 2 ** -8 / 3 ** 0.5, torch.float16: 2 ** -11 / 3 ** 0.5}


def exact(q, k, v, scale, eps=None):
    x = q.double() @ k.double().transpose(-1, -2).contiguous() * scale
    x = x.masked_fill(torch.ones(x.shape[-2:], dtype=torch.bool).triu_(1), float("-inf"))
    w = torch.softmax(x, -1) if eps is None else torch.exp(x)
    den = 1.0 if eps is None else w.sum(-1, keepdim=True).clamp_min(eps)
    return w @ v.double() / den


def rel(a, b):
    return (a.cpu().double() - b).norm().item() / b.norm().item()


# heads x tiles: one workgroup, a full first round, a part of the second, more than two rounds, heads that
# divide by the XCDs and heads that do not; n around the 64- and 32-key batches and the 128-row tiles
@pytest.mark.parametrize("heads,n,d,dv", [
    (1, 1, 4, 4), (1, 63, 64, 64), (2, 64, 16, 16), (3, 65, 40, 72), (1, 129, 128, 128), (2, 257, 33, 30),
    (8, 1025, 64, 64), (8, 4225, 16, 32), (24, 300, 80, 96), (5, 7300, 32, 16), (3, 200, 128, 256), (700, 130, 8, 8),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [0.3, -0.2])
def test_pairs_match_float64(heads, n, d, dv, dtype, scale):
    g = torch.Generator().manual_seed(n * 7 + d)
    q, k, v = (torch.randn(1, heads, n, w, generator=g).mul_(0.7 if w == d else 1.0).to(dtype) for w in (d, d, dv))
    h = torch.tensor(sorted({0, heads // 2, heads - 1}))
    print(heads, n, d, dv, dtype, scale, flush=True)
    out = taa.triton_flash_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=scale)
    ref = exact(q[:, h], k[:, h], v[:, h], scale)
    assert rel(out[:, h.to(DEV)], ref) < (4e-6 if dtype == torch.bfloat16 else 1e-6)
    out = faa.fast_article_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=scale, compressor="none")
    ref = exact(q[:, h], k[:, h], v[:, h], scale, 1e-12)
    assert rel(out[:, h.to(DEV)], ref) < TOL[dtype] + 1e-6


@pytest.mark.parametrize("n,block", [(128, 128), (100, 128), (129, 128)])
def test_sequence_inside_its_first_block(n, block):
    """No coreset item up to n = block: exact attention; past it the block is compressed."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(2, 3, n, 32, generator=g) for _ in range(3))
    out = faa.fast_article_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=0.1, block_size=block)
    ref = exact(q, k, v, 0.1, 1e-12)
    assert rel(out[:, :, :block], ref[:, :, :block]) < (1e-6 if n <= block else 2e-5)  # 2-plane products beyond


@pytest.mark.parametrize("semantics,n,block", [("flat", 100, 128), ("exact", 150, 1)])
def test_clamped_logits_without_items(semantics, n, block):
    """exp_clamp holds where no coreset item takes part: logits up to 120 weigh exp(80), and a logit of 80
    rounds to 2^-17, its weight to 8e-6 of itself."""
    g = torch.Generator().manual_seed(12)
    q, k = (torch.nn.functional.normalize(torch.randn(2, n, 16, generator=g), dim=-1) for _ in range(2))
    k[:, ::9] = q[:, ::9]
    v = torch.randn(2, n, 16, generator=g)
    out = _engine.prefill(q.to(DEV), k.to(DEV), v.to(DEV), degree=2, block=block, scale=120.0, semantics=semantics,
                          exp_clamp=True).out
    x = (q.double() @ k.double().transpose(-1, -2).contiguous() * 120.0).clamp(max=80.0)
    w = torch.exp(x) * torch.ones(n, n, dtype=torch.float64).tril()
    assert rel(out, w @ v.double() / w.sum(-1, keepdim=True)) < 3e-5


def test_pair_weights_and_the_smallest_denominator():
    """Raw weights far below 1 meet the smallest denominator as in num / max(den, eps); scale 0 is the mean."""
    g = torch.Generator().manual_seed(6)
    q = torch.full((1, 2, 70, 16), 2.0)
    k = torch.full((1, 2, 70, 16), -1.5)
    v = torch.randn(1, 2, 70, 16, generator=g)
    out = faa.fast_article_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=1.0, compressor="none",
                                            denominator_eps=1e-3)
    ref = exact(q, k, v, 1.0, 1e-3)
    assert rel(out, ref) < 2 * 48 * 2 ** -24  # the rounding of a logit of -48 is the weight's relative error
    for dtype in (torch.float32, torch.bfloat16):
        out = taa.triton_flash_causal_attention(q.to(DEV, dtype), k.to(DEV, dtype), v.to(DEV, dtype), scale=0.0)
        mean = v.to(dtype).double().cumsum(2) / torch.arange(1, 71).reshape(-1, 1)
        assert rel(out, mean) < 4e-6


# the Taylor part over pairs: chunks of a block (a multiple of 32) and of 32 rows, the level offset of one row,
# row tiles and key batches with remainders, one and several workgroups a tile
@pytest.mark.parametrize("bh,n,d,dv,degree,block", [
    (1, 300, 16, 16, 2, 64), (3, 700, 40, 72, 1, 100), (2, 1153, 64, 64, 2, 128), (64, 385, 32, 32, 3, 96),
    (1, 2049, 128, 128, 2, 256), (2, 260, 20, 200, 0, 50), (9, 513, 7, 30, 3, 37),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("semantics", ["flat", "levels"])
def test_taylor_pairs_match_the_moment_scan(bh, n, d, dv, degree, block, dtype, semantics):
    """Same coreset items and residual, the Taylor part over the pairs or from the moments: each within 5e-6 of
    the sums in 64 bits (split products), plus the rounding of 16-bit outputs."""
    g = torch.Generator().manual_seed(n + d)
    q, k, v = (torch.randn(bh, n, w, generator=g).mul_(s / w ** 0.5).to(dtype).to(DEV)
               for w, s in ((d, 1.0), (d, 1.0), (dv, dv ** 0.5)))
    print(bh, n, d, dv, degree, block, dtype, semantics, flush=True)
    outs = [_engine.prefill(q, k, v, degree=degree, block=block, scale=-0.8, semantics=semantics, moment_kernel=mk,
                            products=pr, out_dtype=torch.float32)
            for mk, pr in (("pairs", None), ("chunked", _native.PRODUCTS_FP32))]
    assert outs[0].moment_kernel == "flash_attn_kernel"
    assert rel(outs[0].out, outs[1].out.cpu().double()) < 5e-6


def _long_pass(dtype, mean):
    """Degree 3 over 65536 keys: the prefill by its kernels, and the last block's rows in 64 bits."""
    n, d, dv, block = 65536, 16, 32, 256
    g = torch.Generator().manual_seed(4)
    q, k = (torch.nn.functional.normalize(torch.randn(1, n, d, generator=g), dim=-1).to(dtype) for _ in range(2))
    v = (torch.randn(1, n, dv, generator=g) + mean).to(dtype)
    run = lambda kernel, products: _engine.prefill(
        q.to(DEV), k.to(DEV), v.to(DEV), degree=3, block=block, scale=1.0, semantics="flat", moment_kernel=kernel,
        residual_products=products, out_dtype=torch.float32)
    res = run("ws", _native.PRODUCTS_FP32)
    poly = lambda x: 1 + x * (1 + x / 2 * (1 + x / 3))
    lo, (q64, k64, v64) = n - block, (x[0].double() for x in (q, k, v))
    x = q64[lo:] @ k64.T.contiguous()
    w = poly(x)
    w[:, lo:] = torch.exp(x[:, lo:]).tril_()
    src = res.node_src[0, :lo // block].flatten().cpu().long()
    xi = q64[lo:] @ k64[src].T.contiguous()
    r = (torch.exp(xi) - poly(xi)) * res.node_w[0, :lo // block].flatten().cpu().double()
    ref = (w @ v64 + r @ v64[src]) / (w.sum(-1) + r.sum(-1))[:, None]
    return lambda kernel, products: (lambda o: (rel(o.out[0, lo:], ref), o.fsplit))(run(kernel, products))


@pytest.mark.parametrize("mean", [0.0, 1.0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_residuals_beside_long_taylor_sums(dtype, mean):
    """The residual kernel's split products drop less than 2^-16 of the residual, a few percent of the weight: with
    either kernel's partial sums they end where the fp32 products end (within half; added to the partials one by one
    the small weights are rounded away, all in one direction: 8 to 20 times the error)."""
    error = _long_pass(dtype, mean)
    for kernel in ("ws", "pairs"):
        assert error(kernel, _native.PRODUCTS_SPLIT_BF16)[0] < 1.5 * error(kernel, _native.PRODUCTS_FP32)[0]


@pytest.mark.parametrize("mean", [0.0, 1.0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_long_taylor_sums_over_pairs(dtype, mean):
    """65536 keys in partial sums of at most 21000 are no further from 64 bits than the scan's sums by features (in
    one sum they are, by a quarter and more)."""
    error = _long_pass(dtype, mean)
    pairs, nsplit = error("pairs", _native.PRODUCTS_FP32)
    assert nsplit == 4
    assert pairs <= error("ws", _native.PRODUCTS_FP32)[0]


def test_pair_rule_and_splits():
    assert _engine.use_pairs(1024, 32, 32, 2, 128)
    assert _engine.use_pairs(4096, 64, 64, 2, 256)
    assert not _engine.use_pairs(65536, 64, 64, 2, 256)
    assert not _engine.use_pairs(3000, 16, 16, 2, 128)
    assert _engine.pair_splits(1, 200, 256) == 1 and _engine.pair_splits(1, 4096, 256) == 8
    assert _engine.pair_splits(64, 4096, 256) == 1


@pytest.mark.parametrize("n,d,dv,dtype", [(1, 64, 64, torch.float32), (127, 16, 30, torch.float16),
                                          (193, 40, 72, torch.bfloat16), (320, 128, 128, torch.float32)])
@pytest.mark.parametrize("products", ["fp32", "split"])
@pytest.mark.parametrize("semantics", ["flat", "levels"])
def test_residual_kernel_inside_one_block(n, d, dv, dtype, products, semantics):
    """Own keys of the residual kernel only (the chunks of 32 rows of the moment scan make the batches in which
    the Taylor part, the residual or both apply): exact attention, to 2e-6 in fp32 products, 1e-5 in split
    products (2^-16 a product), plus the rounding of 16-bit outputs in whole and in partial units."""
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(2, n, w, generator=g).to(dtype) for w in (d, d, dv))
    pr = _native.PRODUCTS_FP32 if products == "fp32" else _native.PRODUCTS_SPLIT_BF16
    print(n, d, dv, dtype, products, semantics, flush=True)
    out = _engine.prefill(q.to(DEV), k.to(DEV), v.to(DEV), degree=2, block=512, scale=0.2, semantics=semantics,
                          products=pr, residual_products=pr, out_dtype=dtype).out
    ref = exact(q, k, v, 0.2, 1e-12)
    assert rel(out, ref) < TOL[dtype] + (2e-6 if products == "fp32" else 1e-5)


@pytest.mark.parametrize("d,dv,block,tokens", [(64, 64, 16, 39), (40, 200, 8, 64), (130, 72, 6, 25), (16, 16, 300, 290)])
@pytest.mark.parametrize("fused", [True, False])
def test_few_streams_tail_matches_many(d, dv, block, tokens, fused):
    """The wide decode tail (up to 256 streams) against the same tokens among 257 streams: fp32 sums in another
    order (a few 2^-23)."""
    g = torch.Generator().manual_seed(d)
    q, k, v = (torch.randn(tokens, 257, w, generator=g).mul_(0.3).to(DEV) for w in (d, d, dv))
    outs = []
    for s in (2, 257):
        att = stc.ArticleStreamingAttention(d, dv, degree=2, block_size=block, streams=s)
        rows = []
        for t in range(tokens):
            if fused:
                rows.append(att.step(q[t, :s], k[t, :s], v[t, :s])[:2])
            else:
                att.update(k[t, :s], v[t, :s])
                rows.append(att.query(q[t, :s])[:2])
        outs.append(torch.stack(rows))
    assert rel(outs[0], outs[1].cpu().double()) < 2e-6


@pytest.mark.parametrize("compressor", ["sorted_pair", "random"])
def test_bulk_draws_ahead_are_bounded(compressor):
    """extend() keeps one upload of draws (64 MiB by its estimate of two calls a completion, half as much again for
    the calls of a run of completions), however many blocks it takes, and draws what single blocks draw."""
    kw = dict(degree=1, block_size=128, streams=2048, compressor=compressor)
    g = torch.Generator(device=DEV).manual_seed(3)
    k, v = (torch.randn(2048, 40 * 128, 8, device=DEV, generator=g) for _ in range(2))
    a, b = (stc.ArticleStreamingAttention(8, 8, **kw) for _ in range(2))
    sizes, draw = [], a._st._draw_completions

    def counted(first, count):
        out = draw(first, count)
        held = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes()
                for dr in list(a._st._draws) + out for t in (dr.methods, dr.dirs, dr.unif, dr.perms)}
        sizes.append(sum(held.values()))
        return out

    a._st._draw_completions = counted
    a.extend(k, v)
    assert len(sizes) > 1 and max(sizes) <= 96 << 20
    for i in range(40):
        b.extend(k[:, 128 * i: 128 * i + 128].contiguous(), v[:, 128 * i: 128 * i + 128].contiguous())
    for x, y in zip(a._st.level_items(), b._st.level_items()):
        assert (x is None) == (y is None)
        assert x is None or all(torch.equal(s, t) for s, t in zip(x, y))


@pytest.mark.parametrize("semantics,bh,n,d,dv,degree,block,dtype,out_dtype", [
    ("flat", 1, 1100, 64, 64, 2, 64, torch.float32, torch.float32), ("flat", 2, 4300, 16, 30, 2, 100, torch.bfloat16, None),
    ("levels", 1, 3000, 40, 72, 2, 48, torch.float16, None), ("levels", 3, 200, 128, 200, 3, 128, torch.float32, None),
    ("segment", 2, 900, 64, 64, 2, 128, torch.float16, torch.float32), ("flat", 1, 700, 200, 16, 2, 64, torch.float32, None),
])
@pytest.mark.parametrize("ksplit", [2, 3, 16])
def test_residual_tiles_shared_by_workgroups(monkeypatch, semantics, bh, n, d, dv, degree, block, dtype, out_dtype, ksplit):
    """ksplit workgroups a tile (more than its batches, and a remainder of its list chunks among them) against
    one: the same terms in another order of fp32 sums (2e-6), rounded to 16 bits at most twice apart."""
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(bh, n, w, generator=g).mul_(0.4).to(dtype).to(DEV) for w in (d, d, dv))
    kw = dict(degree=degree, block=block, scale=0.3, semantics=semantics, stride=2, out_dtype=out_dtype or dtype,
              exp_clamp=semantics == "segment")
    print(semantics, bh, n, d, dv, degree, block, dtype, ksplit, flush=True)
    outs = []
    for s in (1, ksplit):
        monkeypatch.setattr(_engine, "residual_splits", lambda *a, s=s: s)
        outs.append(_engine.prefill(q, k, v, **kw).out)
    assert rel(outs[1], outs[0].cpu().double()) < 2e-6 + 2 * TOL[out_dtype or dtype]


@pytest.mark.parametrize("d,dv", [(16, 16), (8, 5), (32, 16), (128, 16), (256, 12), (24, 24), (64, 32), (256, 32), (256, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_narrow_values_of_the_residual_kernel(d, dv, dtype):
    """Values staged one, two and four keys a thread, own keys and coreset items: split products (2^-16 each) against
    fp32 products, plus the rounding of 16-bit outputs."""
    g = torch.Generator().manual_seed(d + dv)
    q, k, v = (torch.randn(2, 700, w, generator=g).mul_(0.5 if w == d else 1.0).to(dtype).to(DEV) for w in (d, d, dv))
    kw = dict(degree=2, block=48, scale=0.2, semantics="flat", out_dtype=dtype)
    print(d, dv, dtype, flush=True)
    outs = [_engine.prefill(q, k, v, residual_products=pr, **kw).out
            for pr in (_native.PRODUCTS_SPLIT_BF16, _native.PRODUCTS_FP32)]
    assert rel(outs[0], outs[1].cpu().double()) < 2 * TOL[dtype] + 1e-5


def test_residual_split_rule():
    flat = lambda n, block: _engine._plan.flat_plan(n, block, "sorted_pair")
    assert _engine.residual_splits(1, flat(1024, 128), 128, 64, 256) == 1
    assert _engine.residual_splits(1, flat(4096, 256), 256, 128, 256) == 8
    assert _engine.residual_splits(16, flat(3000, 128), 128, 128, 256) == 2
    assert _engine.residual_splits(64, flat(3000, 128), 128, 128, 256) == 1


@pytest.mark.parametrize("heads,n,d,dv,dtype", [(1, 300, 64, 64, torch.float32), (3, 1025, 40, 72, torch.bfloat16),
                                                (2, 130, 128, 200, torch.float16), (8, 65, 16, 5, torch.float32)])
@pytest.mark.parametrize("nsplit", [2, 5, 8])
def test_exact_tiles_shared_by_workgroups(monkeypatch, heads, n, d, dv, dtype, nsplit):
    """nsplit workgroups a tile, more than its key batches among them, against float64 (bounds as above)."""
    monkeypatch.setattr(_engine, "flash_splits", lambda *a: nsplit)
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(1, heads, n, w, generator=g).to(dtype) for w in (d, d, dv))
    out = taa.triton_flash_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=0.4)
    assert rel(out, exact(q, k, v, 0.4)) < (4e-6 if dtype == torch.bfloat16 else 1e-6)
    out = faa.fast_article_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=0.1, compressor="none")
    assert rel(out, exact(q, k, v, 0.1, 1e-12)) < TOL[dtype] + 1e-6


MASKS = {"lowest": torch.finfo(torch.float32).min, "-inf": float("-inf")}


@pytest.mark.parametrize("heads,n,d,dv,nsplit", [(2, 40, 16, 16, 1), (1, 300, 33, 72, 1), (3, 1025, 64, 64, 5),
                                                 (1, 130, 128, 200, 2)])
@pytest.mark.parametrize("mask", sorted(MASKS))
def test_keys_switched_off_by_a_dimension(monkeypatch, heads, n, d, dv, nsplit, mask):
    """A key dimension of the type's lowest value or -inf against queries of 1 there: weight 0 for those keys, also
    for rows that have seen no other key, whose sums are then 0.  fp32 products (1e-6)."""
    monkeypatch.setattr(_engine, "flash_splits", lambda *a: nsplit)
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(1, heads, n, w, generator=g) for w in (d, d, dv))
    q[..., 0], k[..., 0] = 1.0, 0.0
    k[:, :, 5::7, 0] = MASKS[mask]
    k[:, :, :2, 0] = MASKS[mask]
    print(heads, n, d, dv, nsplit, mask, flush=True)
    out = taa.triton_flash_causal_attention(q.to(DEV), k.to(DEV), v.to(DEV), scale=0.4)
    assert (out[:, :, :2] == 0).all()
    assert rel(out[:, :, 2:], exact(q, k, v, 0.4)[:, :, 2:]) < 1e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,d,dv,nsplit", [(300, 64, 64, 1), (700, 16, 40, 3)])
def test_infinite_and_largest_values(monkeypatch, dtype, n, d, dv, nsplit):
    """An infinite value makes its column infinite from its row on and leaves the columns beside it, and rows at
    least a key batch before it, as they are; the largest finite value stays finite under softmax weights."""
    monkeypatch.setattr(_engine, "flash_splits", lambda *a: nsplit)
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(1, 2, n, w, generator=g).to(dtype) for w in (d, d, dv))
    at = n // 2 // 64 * 64 + 3
    vi = v.clone()
    vi[:, :, at, 3] = float("inf")
    if dtype != torch.float32:  # the two-plane 16-bit weights of the softmax make inf or NaN of it
        fns = [(lambda x: faa.fast_article_causal_attention(*x, scale=0.1, compressor="none"), 0.1, 1e-12)]
    else:
        fns = [(lambda x: faa.fast_article_causal_attention(*x, scale=0.1, compressor="none"), 0.1, 1e-12),
               (lambda x: taa.triton_flash_causal_attention(*x, scale=0.1), 0.1, None)]
    print(n, d, dv, nsplit, dtype, flush=True)
    for fn, scale, eps in fns:
        out = fn([x.to(DEV) for x in (q, k, vi)]).cpu()
        ref = exact(q, k, v, scale, eps)
        assert (out[:, :, at:, 3] == float("inf")).all()
        keep = torch.ones(n, dv, dtype=torch.bool)
        keep[at - 63:, 3] = False
        assert rel(out[:, :, keep], ref[:, :, keep]) < TOL[dtype] + 1e-6
    vm = v.clone()
    vm[:, :, at, 3] = torch.finfo(dtype).max
    out = taa.triton_flash_causal_attention(*(x.to(DEV) for x in (q, k, vm)), scale=0.1).cpu()
    ref = exact(q, k, vm, 0.1)
    rest = torch.arange(dv) != 3
    tol = 4e-6 if dtype == torch.bfloat16 else 1e-6
    assert rel(out[:, :, at:, 3] * 2.0 ** -100, ref[:, :, at:, 3] * 2.0 ** -100) < tol
    assert rel(out[..., rest], ref[..., rest]) < tol


@pytest.mark.parametrize("power", [-100, -118])
def test_tiny_values_keep_their_bits(power):
    """Values whose lower planes would be subnormal: linear in the values, so 1e-6 as at ordinary sizes."""
    g = torch.Generator().manual_seed(8)
    q, k, v = (torch.randn(1, 2, 200, 32, generator=g) for _ in range(3))
    out = taa.triton_flash_causal_attention(q.to(DEV), k.to(DEV), (v * 2.0 ** power).to(DEV), scale=0.3)
    assert rel(out.cpu().double() * 2.0 ** -power, exact(q, k, v, 0.3)) < 1e-6


@pytest.mark.parametrize("dtype,ld", [(torch.float32, 1 << 27), (torch.bfloat16, 1 << 28)])
def test_row_strides_beyond_a_batch_buffer(dtype, ld):
    """Rows 512 MiB apart (q, k and v side by side in one allocation): the batch offsets leave the 1 GiB buffers."""
    n, d, dv = 3, 16, 8
    big = torch.empty(n, ld, device=DEV, dtype=dtype)
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(1, 1, n, w, generator=g).to(dtype) for w in (d, d, dv))
    for i, x in enumerate((q, k, v)):
        big[:, 16 * i: 16 * i + x.shape[-1]] = x[0, 0].to(DEV)
    out = torch.empty(n, dv, device=DEV)
    lib, es = _native.lib(), big.element_size()
    print(dtype, ld, flush=True)
    _native.check(lib.sta_flash_attention(big.data_ptr(), big.data_ptr() + 16 * es, big.data_ptr() + 32 * es,
                                          _native.DTYPE_CODES[dtype], 1, n, d, dv, ld, ld, 0.3, out.data_ptr(),
                                          _native.DTYPE_CODES[torch.float32],
                                          _native.stream_handle(torch.device(DEV))), "sta_flash_attention")
    assert rel(out, exact(q, k, v, 0.3)[0, 0]) < 1e-6


def test_exact_split_rule():
    sp = lambda bh, n, w=64: _engine.flash_splits(bh, n, w, w, 256)
    assert [sp(1, 8192), sp(4, 8192), sp(8, 8191), sp(32, 2048), sp(40, 2048), sp(64, 1024), sp(1, 500, 32)] == \
        [8, 4, 3, 2, 1, 1, 1]


def test_splits_that_would_cost_more_than_they_give():
    """The second launch and the partial sums' traffic: short 16-bit tiles, wide rows in many tiles."""
    b16, f16, f32 = torch.bfloat16, torch.float16, torch.float32
    sp = lambda bh, n, w, dt, softmax=True: _engine.flash_splits(bh, n, w, w, 256, dt, softmax)
    assert [sp(4, 500, 64, b16), sp(32, 700, 64, f16), sp(64, 512, 128, b16), sp(64, 512, 128, f32), sp(32, 2048, 64, b16),
            sp(4, 500, 64, f32, False), sp(4, 500, 64, b16, False), sp(32, 700, 64, f16, False)] == [1] * 8
    assert sp(4, 500, 64, f32) > 1 and sp(1, 1500, 16, f32) > 1 and sp(4, 8192, 64, b16) > 1
    assert sp(32, 1000, 64, f16, False) > 1 and sp(4, 1500, 64, b16, False) > 1 and sp(32, 2048, 64, b16, False) > 1
    flat = lambda n, block: _engine._plan.flat_plan(n, block, "sorted_pair")
    levels = lambda n, block: _engine._plan.levels_plan(n, block, "sorted_pair")
    assert _engine.residual_splits(64, flat(450, 128), 128, 256, 256) == 1
    assert _engine.residual_splits(48, flat(1000, 128), 128, 128, 256) == 1
    assert _engine.residual_splits(16, levels(3000, 128), 128, 128, 256) == 1
    assert _engine.residual_splits(1, levels(4096, 256), 256, 128, 256) > 1
