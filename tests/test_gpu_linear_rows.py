"""Products of 1 to 64 rows with the step after them (``kernels.linear_rows``) against float64 references: row
tiles that are whole and not, one and two halves of the rows, half tiles of the weights (up to 16 rows, where tiles are few), one to
three tiles a workgroup, K that gives the eight waves unequal shares or none, bfloat16 and (up to 16 rows) float32; and the
attention kernels that write their rows in the order these products read."""

import pytest
import torch

import plain_llama as P
from test_gpu_kernels import DEV, K, _bf, read_cache, rnd

pytestmark = pytest.mark.gpu


# Tiles of W at most half the CUs (2,048 columns and below): two workgroups share the rows beyond 16, or a tile of the weights up to
# 16 rows; more (4,096): one, or two halves of the rows.
@pytest.mark.parametrize("n,m,k", [(1, 16, 32), (17, 48, 96), (5, 64, 2048), (8, 2048, 5632), (3, 72, 448), (9, 40, 64), (16, 2048, 2048), (12, 1000, 1152), (16, 4096, 320), (33, 72, 288), (45, 2048, 2048), (48, 100, 5632),
                                   (64, 2048, 5632), (64, 4096, 1056), (50, 4096, 4096), (32, 1000, 736), (63, 4090, 160)])
def test_resid_then_scaled_consumers(n, m, k):
    """The product added to the residual stream, what the norm behind it needs left beside it, and the two
    consumers that scale their sums.  Bounds as for the decode-batch kernel's test: sums of k products of 16-bit
    operands in 32 bits, xw and the consumers' results rounded to 16 bits."""
    k_, eps = K(), 1e-5
    x, w = _bf(n, k, seed=1, scale=0.5), _bf(m, k, seed=2, scale=0.1)
    resid, nw = rnd(n, m, seed=3, scale=2.0), 1 + 0.2 * rnd(m, seed=4)
    parts = k_.linear_rows_parts(n, m, k)
    ss = torch.full((n, -(-parts // 4) * 4), float("nan"), device=DEV)
    xw = torch.full((n, m), float("nan"), dtype=torch.bfloat16, device=DEV)
    stream = resid.clone()
    k_.linear_rows(k_.fused_linear_tile(w, k_.LINEAR_PARTS), xw, k_.LINEAR_RESID, x, resid=stream, norm_weight=nw, ss_out=ss)
    want_x = resid.double() + x.double() @ w.double().T
    assert (stream.double() - want_x).abs().max() < 1e-3 * k ** 0.5 * 0.05 + 1e-4
    assert (xw.double() - want_x * nw.double()).abs().max() < 0.005 * want_x.abs().max() * 1.2 + 1e-3
    got_ss = ss[:, :parts].double().sum(1)
    assert ((got_ss - (want_x ** 2).sum(1)).abs() / (want_x ** 2).sum(1)).max() < 1e-4
    if m % 32:
        return
    want_n = P.rmsnorm(want_x, nw.double(), eps)
    # the same rows in the order that the next product's lanes read them: the same bits
    xt = k_.TiledRows(torch.full((k_.TiledRows.stored(n), m), float("nan"), dtype=torch.bfloat16, device=DEV), n)
    stream2, ss2 = resid.clone(), torch.zeros_like(ss)
    k_.linear_rows(k_.fused_linear_tile(w, k_.LINEAR_PARTS), xt, k_.LINEAR_RESID, x, resid=stream2, norm_weight=nw, ss_out=ss2)
    assert torch.equal(stream2, stream) and torch.equal(ss2[:, :parts], ss[:, :parts])
    sr, st = k_.ScaledRows(xw, ss, parts, eps), k_.ScaledRows(xt, ss, parts, eps)
    for f in (32, 40, 2056, 3080):      # one tile to a workgroup (4 and 5 of them), two (257 x 2), two (385)
        wg = _bf(2 * f, m, seed=5, scale=0.1)
        h = torch.full((n, f), float("nan"), dtype=torch.bfloat16, device=DEV)
        k_.linear_rows(k_.fused_linear_tile(wg, k_.LINEAR_SWIGLU), h, k_.LINEAR_SWIGLU, sr)
        g = want_n @ wg[:f].double().T
        want = g * torch.sigmoid(g) * (want_n @ wg[f:].double().T)
        assert (h.double() - want).abs().max() < 0.01 * want.abs().max() + 2e-3
        h2 = torch.full_like(h, float("nan"))
        k_.linear_rows(k_.fused_linear_tile(wg, k_.LINEAR_SWIGLU), h2, k_.LINEAR_SWIGLU, st)
        assert torch.equal(h2, h)
        if f % 32 == 0:                 # a tiled output as the next product's input
            wn = _bf(96, f, seed=9, scale=0.1)
            ht = k_.TiledRows(torch.full((k_.TiledRows.stored(n), f), float("nan"), dtype=torch.bfloat16, device=DEV), n)
            k_.linear_rows(k_.fused_linear_tile(wg, k_.LINEAR_SWIGLU), ht, k_.LINEAR_SWIGLU, st)
            got = []
            for hin in (h, ht):
                z, y, zs = torch.zeros(n, 96, device=DEV), torch.empty(n, 96, dtype=torch.bfloat16, device=DEV), None
                zs = torch.empty(n, -(-k_.linear_rows_parts(n, 96, f) // 4) * 4, device=DEV)
                k_.linear_rows(k_.fused_linear_tile(wn, k_.LINEAR_PARTS), y, k_.LINEAR_RESID, hin, resid=z,
                               norm_weight=torch.ones(96, device=DEV), ss_out=zs)
                got.append((z, y))
            assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    H, hd = 2, 16
    wq = _bf(H * hd, m, seed=6, scale=0.1)
    pos = torch.arange(5, 5 + n, dtype=torch.int32, device=DEV)
    cos, sin = torch.empty(n, hd // 2, device=DEV), torch.empty(n, hd // 2, device=DEV)
    k_.rope_tables(cos, sin, pos, hd, 10000.0)
    q = torch.full((n, H * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    rope = k_.Rope(cos, sin, None, None, None, None, 16, H, 1, hd)
    k_.linear_rows(k_.fused_linear_tile(wq, k_.LINEAR_ROPE, rope), q, k_.LINEAR_ROPE, sr, rope=rope)
    want_q = P.rope((want_n @ wq.double().T).cpu(), pos.cpu().tolist(), H, hd, 10000.0)
    assert (q.cpu().double() - want_q).abs().max() < 0.01 * want_q.abs().max() + 2e-3


@pytest.mark.parametrize("n,f,k", [(64, 5632, 2048), (45, 5632, 512), (33, 24, 64), (17, 3000, 1024), (61, 4104, 320),
                                   (31, 6000, 96)])
def test_swiglu_of_a_strided_view(n, f, k):
    """Up to three tiles a workgroup (5,632 and 6,000: 704 and 750 tiles), the last group not whole."""
    k_ = K()
    x, w = _bf(n, k + 24, seed=7, scale=0.5)[:, 8:8 + k], _bf(2 * f, k, seed=8, scale=0.1)
    h = torch.full((n, f), float("nan"), dtype=torch.bfloat16, device=DEV)
    k_.linear_rows(k_.fused_linear_tile(w, k_.LINEAR_SWIGLU), h, k_.LINEAR_SWIGLU, x, act=k_.ACT_GELU_TANH)
    xd, wd = x.double(), w.double()
    want = torch.nn.functional.gelu(xd @ wd[:f].T, approximate="tanh") * (xd @ wd[f:].T)
    assert (h.double() - want).abs().max() < 0.01 * want.abs().max() + 1e-3


@pytest.mark.parametrize("n,f,k,dtype", [(8, 6200, 96, "bfloat16"), (3, 6200, 2048, "bfloat16"), (13, 6200, 2080, "bfloat16"),
                                         (16, 6152, 4096, "bfloat16"), (33, 6200, 64, "bfloat16"), (2, 6152, 96, "float32"),
                                         (11, 6200, 96, "float32"), (16, 6152, 2048, "float32")])
def test_swiglu_of_more_than_three_tiles_a_cu(n, f, k, dtype):
    """769 and 775 tiles: two a workgroup, one where K is long, the last group not whole; rows as they are and in the lanes' order
    (16 rows of 4,096 go one tile a workgroup only there) give the same bits.  Bounds: 16-bit results of 32-bit sums; in float32
    a sum of k products of 0.05 has an error of 2^-24 sqrt(k) of its size, and the gate multiplies two of them."""
    k_, dt = K(), getattr(torch, dtype)
    x, w = rnd(n, k, seed=1, scale=0.5).to(dt), rnd(2 * f, k, seed=2, scale=0.1).to(dt)
    tiled = k_.fused_linear_tile(w, k_.LINEAR_SWIGLU)
    h = torch.full((n, f), float("nan"), dtype=dt, device=DEV)
    k_.linear_rows(tiled, h, k_.LINEAR_SWIGLU, x)
    g = x.double() @ w[:f].double().T
    want = g * torch.sigmoid(g) * (x.double() @ w[f:].double().T)
    if dtype == "float32":
        assert (h.double() - want).abs().max() < 1e-5 * (g.abs().max() ** 2 + 1)
        return
    assert (h.double() - want).abs().max() < 0.01 * want.abs().max() + 2e-3
    xt = k_.TiledRows(torch.zeros(k_.TiledRows.stored(n), k, dtype=dt, device=DEV), n)
    for r in range(n):
        for_row = xt.data.view(-1, k // 32, 4, min(n, 16), 8)[r // 16, :, :, r % 16]
        for_row.copy_(x[r].view(k // 32, 4, 8))
    k_.linear_rows(tiled, h2 := torch.full_like(h, float("nan")), k_.LINEAR_SWIGLU, xt)
    assert torch.equal(h2, h)


@pytest.mark.parametrize("H,KV,hd,ps,d", [(4, 2, 16, 16, 64), (5, 5, 48, 32, 96), (32, 4, 64, 16, 2048), (3, 3, 80, 16, 128)])
def test_rope_append(H, KV, hd, ps, d):
    """Projections, rotation and append of 40 tokens of four requests."""
    k_, theta = K(), 10000.0
    spans = [(ps - 3, 13), (0, 9), (ps - 1, 1), (5, 17)]
    n = sum(l for _, l in spans)
    pos = torch.tensor([p0 + i for p0, l in spans for i in range(l)], dtype=torch.int32, device=DEV)
    sot = torch.tensor([s for s, (_, l) in enumerate(spans) for _ in range(l)], dtype=torch.int32, device=DEV)
    tables = [[9, 4], [2, 1], [7, -1], [3, 0]]
    bt = torch.tensor(tables, dtype=torch.int32, device=DEV)
    qd, kvd = H * hd, KV * hd
    x, w = _bf(n, d, seed=3, scale=0.5), _bf(qd + 2 * kvd, d, seed=4, scale=0.1)
    cos, sin = torch.empty(n, hd // 2, device=DEV), torch.empty(n, hd // 2, device=DEV)
    k_.rope_tables(cos, sin, pos, hd, theta)
    cache = torch.full((12, 2, KV, ps * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    q_out = torch.full((n, qd), float("nan"), dtype=torch.bfloat16, device=DEV)
    rope = k_.Rope(cos, sin, cache, pos, sot, bt, ps, H, KV, hd)
    k_.linear_rows(k_.fused_linear_tile(w, k_.LINEAR_ROPE, rope), q_out, k_.LINEAR_ROPE, x, rope=rope)
    full = P.linear(x.cpu().double(), w.cpu().double())
    want_q = P.rope(full[:, :qd], pos.cpu().tolist(), H, hd, theta)
    want_k = P.rope(full[:, qd:qd + kvd], pos.cpu().tolist(), KV, hd, theta)
    t = 0.01 * full.abs().max() + 1e-3
    assert (q_out.cpu().double() - want_q).abs().max() < t
    off = 0
    for s, (p0, l) in enumerate(spans):
        ks, vs = read_cache(cache, tables[s], p0 + l, KV, hd, ps)
        assert (ks[p0:].double() - want_k[off:off + l]).abs().max() < t
        assert (vs[p0:].double() - full[off:off + l, qd + kvd:]).abs().max() < t
        assert torch.isnan(ks[:p0]).all() and torch.isnan(vs[:p0]).all()
        off += l


def test_refusals():
    k_ = K()
    w = _bf(64, 96, seed=1, scale=0.1)
    tiled = k_.fused_linear_tile(w, k_.LINEAR_SWIGLU)
    h = torch.empty(20, 32, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(k_.KernelError, match="tiled copy"):
        k_.linear_rows(w, h, k_.LINEAR_SWIGLU, _bf(20, 96, seed=2, scale=1.0))
    with pytest.raises(k_.KernelError, match="outside"):
        k_.linear_rows(tiled, torch.empty(65, 32, dtype=torch.bfloat16, device=DEV), k_.LINEAR_SWIGLU, _bf(65, 96, seed=2, scale=1.0))
    with pytest.raises(k_.KernelError, match="multiple of 32"):
        k_.linear_rows(k_.fused_linear_tile(_bf(64, 40, seed=1, scale=0.1), k_.LINEAR_SWIGLU), h, k_.LINEAR_SWIGLU,
                       _bf(20, 40, seed=2, scale=1.0))


@pytest.mark.parametrize("n,m,k", [(1, 40, 64), (8, 2048, 2048), (5, 72, 96), (13, 2048, 1536), (16, 5632, 2048), (20, 5632, 512),
                                   (33, 4096, 1056), (64, 2048, 5632), (45, 12300, 160), (3, 9000, 544), (45, 12200, 160),
                                   (20, 8400, 96), (64, 12288, 64)])
def test_sums_and_activations_of_them(n, m, k):
    """Plain sums, and an activation of them in 16 bits: half tiles of W, whole ones, two (5,632 columns) and three (8,400 to 12,288)
    a workgroup, and one of 769 tiles (12,300)."""
    k_ = K()
    x, w = _bf(n, k, seed=1, scale=0.5), _bf(m, k, seed=2, scale=0.1)
    tiled = k_.fused_linear_tile(w, k_.LINEAR_PARTS)
    want = x.double() @ w.double().T
    y = torch.full((1, n, m), float("nan"), device=DEV)
    k_.linear_rows(tiled, y, k_.LINEAR_PARTS, x)
    assert (y[0].double() - want).abs().max() < 1e-3 * k ** 0.5 * 0.05 + 1e-4      # (as for the decode-batch kernel's sums)
    h = torch.full((n, m), float("nan"), dtype=torch.bfloat16, device=DEV)
    k_.linear_rows(tiled, h, k_.LINEAR_PARTS, x, unary=(k_.ACT_RELU_SQ, None))
    want = want.clamp(min=0) ** 2
    assert (h.double() - want).abs().max() < 0.01 * want.abs().max() + 1e-3
    params = torch.tensor([0.3, -0.2], device=DEV)
    k_.linear_rows(tiled, h, k_.LINEAR_PARTS, x, unary=(k_.ACT_XIELU, params))
    k_.unary_act(y, h2 := torch.empty_like(h), k_.ACT_XIELU, params)
    assert torch.equal(h, h2)


def _rowwise(t):
    """TiledRows as plain rows."""
    n, k = t.shape
    side = min(n, 16)
    v = t.data.reshape(-1, k // 32, 4, side, 8)[: -(-n // 16)]
    return v.permute(0, 3, 1, 2, 4).reshape(-1, k)[:n]


@pytest.mark.parametrize("H,KV,hd,ps", [(8, 2, 16, 16), (32, 4, 64, 16), (6, 6, 128, 32)])
@pytest.mark.parametrize("slices", [1, 4, 33])
def test_attention_writes_tiled_rows(H, KV, hd, ps, slices):
    """Decode attention (one workgroup and merged slices) and prompt attention write the same numbers in the
    order that the output projection's lanes read."""
    k_ = K()
    for spans in ([(9, 1), (70, 1), (300, 1)], [(5, 1)] * 16, [(0, 37), (130, 3)]):
        n = sum(l for _, l in spans)
        pages = [-(-(p0 + l) // ps) for p0, l in spans]
        bt = torch.zeros(len(spans), max(pages), dtype=torch.int32)
        at = 0
        for i, c in enumerate(pages):
            bt[i, :c] = torch.arange(at, at + c)
            at += c
        bt = bt.to(DEV)
        cache, q = _bf(at, 2, KV, ps * hd, seed=1, scale=1.0), _bf(n, H * hd, seed=2, scale=1.0)
        pos = torch.tensor([p0 + i for p0, l in spans for i in range(l)], dtype=torch.int32, device=DEV)
        sot = torch.tensor([s for s, (_, l) in enumerate(spans) for _ in range(l)], dtype=torch.int32, device=DEV)
        part = torch.empty(n * H * slices * (hd + 2), device=DEV)
        out = torch.empty(n, H * hd, dtype=torch.bfloat16, device=DEV)
        tiled = k_.TiledRows(torch.zeros(k_.TiledRows.stored(n), H * hd, dtype=torch.bfloat16, device=DEV), n)
        for o in (out, tiled):
            k_.attn_decode(q, o, part, cache, pos, sot, bt, ps, H, KV, hd, 0, hd ** -0.5, slices)
        assert torch.equal(_rowwise(tiled), out)
        if hd in k_.PREFILL_HEAD_DIMS and slices == 1:
            start = torch.tensor([0] + torch.tensor([l for _, l in spans]).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
            tiles = torch.tensor([[int(start[s]), s] for s in range(len(spans))], dtype=torch.int32, device=DEV)
            span_pos = torch.tensor([p0 for p0, _ in spans], dtype=torch.int32, device=DEV)
            for keys in (0, 10 ** 6):            # both kernels
                for o in (out, tiled):
                    k_.attn_prefill(q, o, cache, tiles, len(spans), start, span_pos, bt, ps, H, KV, hd, 0, hd ** -0.5,
                                    keys, keys)
                assert torch.equal(_rowwise(tiled), out)
            most = k_.attn_prefill_slices(len(spans), H, hd)
            assert (most > 1) == (hd == 128)
            if most > 1:                         # the blocks' keys in slices, merged in the same call
                part = torch.full((n * H * most * (hd + 2),), float("nan"), device=DEV)
                out2 = torch.zeros_like(out)
                tiled.data.zero_()
                for o in (out2, tiled):
                    k_.attn_prefill(q, o, cache, tiles, len(spans), start, span_pos, bt, ps, H, KV, hd, 0, hd ** -0.5,
                                    10 ** 6, 10 ** 6, part=part, nslices=most)
                # (16-bit results, the slices' sums in 32: one rounding apart)
                assert torch.equal(_rowwise(tiled), out2) and (out2 - out).abs().max() <= 2.0 ** -7 * out.abs().max()


@pytest.mark.parametrize("n,m,k", [(5, 64, 64), (8, 2048, 2048), (8, 2048, 5632), (13, 72, 448), (16, 2048, 5632), (16, 4096, 4096),
                                   (7, 4096, 1056), (1, 40, 32)])
def test_float32(n, m, k):
    """True 32-bit products and the steps after them: sums as close to 64 bits as the decode-batch kernel's."""
    k_, f32, eps = K(), torch.float32, 1e-5
    x, w = rnd(n, k, seed=1, scale=0.5), rnd(m, k, seed=2, scale=0.1)
    tiled = k_.fused_linear_tile(w, k_.LINEAR_PARTS)
    want = x.double() @ w.double().T
    y, y2 = torch.full((1, n, m), float("nan"), device=DEV), torch.empty(1, n, m, device=DEV)
    k_.linear_rows(tiled, y, k_.LINEAR_PARTS, x)
    k_.fused_linear(tiled, y2, k_.LINEAR_PARTS, x)
    k_.linear_rows(w, y3 := torch.empty_like(y), k_.LINEAR_PARTS, x)
    assert torch.equal(y3, y)                       # from the matrix itself
    # products of 0.5 x 0.1 added k at a time: 32-bit chains of at most k / 64 and 64 of them in a tree
    bound = 0.05 * k ** 0.5 * 2.0 ** -24 * 8
    assert (y[0].double() - want).norm() <= 1.1 * (y2[0].double() - want).norm() + 1e-12
    assert (y[0].double() - want).abs().max() < 6 * bound + 1e-7
    resid, nw = rnd(n, m, seed=3, scale=2.0), 1 + 0.2 * rnd(m, seed=4)
    parts = k_.linear_rows_parts(n, m, k)
    ss = torch.full((n, -(-parts // 4) * 4), float("nan"), device=DEV)
    stream, xw = resid.clone(), torch.empty(n, m, device=DEV)
    k_.linear_rows(tiled, xw, k_.LINEAR_RESID, x, resid=stream, norm_weight=nw, ss_out=ss)
    want_x = resid.double() + want
    assert (stream.double() - want_x).abs().max() < 6 * bound + 1e-6
    assert torch.equal(xw, stream * nw)
    k_.linear_rows(w, xw, k_.LINEAR_RESID, x, resid=(stream2 := resid.clone()), norm_weight=nw, ss_out=ss)
    assert torch.equal(stream2, stream)
    assert ((ss[:, :parts].double().sum(1) - (want_x ** 2).sum(1)).abs() / (want_x ** 2).sum(1)).max() < 1e-5
    if m % 32:
        return
    want_n, sr = P.rmsnorm(want_x, nw.double(), eps), k_.ScaledRows(xw, ss, parts, eps)
    for f in (40, 2056, 3080):
        wg = rnd(2 * f, m, seed=5, scale=0.1)
        h = torch.full((n, f), float("nan"), device=DEV)
        k_.linear_rows(k_.fused_linear_tile(wg, k_.LINEAR_SWIGLU), h, k_.LINEAR_SWIGLU, sr)
        k_.linear_rows(wg, h2 := torch.empty_like(h), k_.LINEAR_SWIGLU, sr)
        assert torch.equal(h2, h)
        g = want_n @ wg[:f].double().T
        assert ((h.double() - g * torch.sigmoid(g) * (want_n @ wg[f:].double().T)).abs().max()
                < 1e-5 * (g.abs().max() ** 2 + 1))
    H, hd = 2, 16
    wq = rnd(H * hd, m, seed=6, scale=0.1)
    pos = torch.arange(5, 5 + n, dtype=torch.int32, device=DEV)
    cos, sin = torch.empty(n, hd // 2, device=DEV), torch.empty(n, hd // 2, device=DEV)
    k_.rope_tables(cos, sin, pos, hd, 10000.0)
    rope, q = k_.Rope(cos, sin, None, None, None, None, 16, H, 1, hd), torch.full((n, H * hd), float("nan"), device=DEV)
    k_.linear_rows(k_.fused_linear_tile(wq, k_.LINEAR_ROPE, rope), q, k_.LINEAR_ROPE, sr, rope=rope)
    k_.linear_rows(wq, q2 := torch.empty_like(q), k_.LINEAR_ROPE, sr, rope=rope)
    assert torch.equal(q2, q)
    want_q = P.rope((want_n @ wq.double().T).cpu(), pos.cpu().tolist(), H, hd, 10000.0)
    assert (q.cpu().double() - want_q).abs().max() < 1e-5 * (want_q.abs().max() + 1)


@pytest.mark.parametrize("m,k", [(16, 32), (100, 64), (513, 512), (2048, 2048), (1030, 1056), (16383, 96)])
def test_plain_sums_of_a_decode_batch_by_either_kernel(m, k):
    """``decode_linear`` up to 16 rows from the tiled copy, rows apart by more than K among them: against the decode-batch kernel
    (the option that keeps products from the library leaves it that one) and the product in 64 bits.  A sum's error is at most K
    units of the 32-bit rounding of the sum of magnitudes, either way; an activation rounds to bfloat16 behind it."""
    from types import SimpleNamespace
    from kllm_amd.parts import linear as products
    k_ = K()
    ctx = [SimpleNamespace(runtime=SimpleNamespace(options=o, dtype=torch.bfloat16),
                           buf=lambda tag, shape, dtype: torch.full(shape, float("nan"), dtype=dtype, device=DEV)) for o in ({}, {"gemm": "library"})]
    w = _bf(m, k, seed=3, scale=0.1)
    tiled = k_.fused_linear_tile(w, k_.LINEAR_PARTS)
    for n in (1, 2, 8, 9, 15, 16):
        for x in (_bf(n, k, seed=n, scale=1.0), _bf(n, k + 40, seed=n, scale=1.0)[:, 8:k + 8]):
            assert products._unstaged(ctx[0].runtime, n, m, k, x.dtype, tiled) and not products._unstaged(ctx[1].runtime, n, m, k, x.dtype, tiled)
            ref = x.double() @ w.double().T
            bound = k * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T)
            for c in ctx:
                assert ((products.decode_linear(c, x, w, "y", tiled).double() - ref).abs() <= bound).all(), (n, x.stride(0))
                h = products.decode_linear(c, x, w, "h", tiled, unary=(k_.ACT_RELU_SQ, None)).double()
                want = ref.clamp_min(0) ** 2
                assert ((h - want).abs() <= 2.0 ** -8 * want + (2 * ref.abs() + bound) * bound * 1.01).all(), (n, x.stride(0))
