"""The rules that choose a product's tile and its slices of K: plain host code, checked without a GPU
(the library counts 256 CUs where it cannot ask)."""

import types

import pytest
import torch

from kllm_amd import kernels as K
from kllm_amd.engine.engine import room_for_copies
from kllm_amd.parts import linear as products
from kllm_amd.parts.base import ResidualSink
from kllm_amd.parts.linear import choose
from kllm_amd.parts.recurrent import takes_sixteens

BF16, F32 = torch.bfloat16, torch.float32
LONG = 1 << 23          # from this K on a lane's offset takes 64 bits


@pytest.mark.parametrize("n,m,k,dtype,slices", [
    (65, 3, LONG + 8, BF16, 8), (2000, 4096, LONG, BF16, 8), (2, 3, LONG + 8, F32, 8), (65, 3, LONG + 4, F32, 8),
    (64, 3, LONG + 8, BF16, 1), (2, 3, LONG + 8, BF16, 1), (64, 2048, 5632, BF16, 1), (1, 8, 8, BF16, 1),
    (0, 8, 8, BF16, 1),
])
def test_slices_where_the_times_are_not_estimated(n, m, k, dtype, slices):
    """Also right behind a product whose times are, which leaves its numbers on the stack."""
    for other in ((700, 2048, 5632), (64, 2048, 5632), (2048, 28672, 4096)):
        K.gemm_prompt_slices(*other, dtype)
        K.gemm_prompt_slices.cache_clear()
        assert K.gemm_prompt_slices(n, m, k, dtype) == slices


@pytest.mark.parametrize("n", [9, 17, 33, 48, 49, 64, 65, 128, 700, 2048])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_no_slice_of_k_is_empty(n, dtype):
    """The MFMA tiles round a slice up to two stages (256 bytes of K), or to one where that leaves the last slice
    empty; the skinny kernel up to 32: with the kernel's own rounding the last slice must hold something, for the
    widths of the models here and for K around every multiple of those."""
    each = 8 if dtype == BF16 else 4
    ks = {k + d * each for k in (64, 512, 1024, 2048, 4096, 5632, 7168, 11008, 14336) for d in (-9, -1, 0, 1, 5)}
    cut = 0
    for m in (256, 1000, 2048, 2560, 4096, 11264, 28672):
        for k in sorted(ks):
            if k <= 0:
                continue
            algo, nsplit = choose(dtype, n, m, k)
            if algo not in (K.GEMM_MFMA_BF16, K.GEMM_MFMA_F32, K.GEMM_SKINNY_BF16):
                continue
            unit = 32 if algo == K.GEMM_SKINNY_BF16 else 256 // (16 // each)
            kslice = -(-(-(-k // nsplit)) // unit) * unit
            if algo != K.GEMM_SKINNY_BF16 and (nsplit - 1) * kslice >= k:
                kslice = -(-(-(-k // nsplit)) // (unit // 2)) * (unit // 2)
            assert (nsplit - 1) * kslice < k, (m, k, nsplit, kslice)
            cut += nsplit > 1
    assert cut


@pytest.mark.parametrize("n,m,k,dtype,slices", [
    (17, 2048, 5632, F32, 16), (64, 2048, 5632, F32, 16),            # (of 352; of 384 the last one would be empty)
    (17, 2048, 5640, BF16, 10), (48, 2040, 7176, BF16, 13),          # (of 576, not 640)
    (17, 2048, 5632, BF16, 11), (49, 2048, 5632, BF16, 8), (17, 4096, 5632, BF16, 8),
])
def test_slices_of_a_decode_batch(n, m, k, dtype, slices):
    assert choose(dtype, n, m, k)[1] == slices


@pytest.mark.parametrize("weights,cache,free,total,room", [
    (4, 1, 280, 288, True), (32, 80, 250, 288, True), (32, 81, 250, 288, False),    # half of the card stays
    (32, 230, 250, 288, False), (100, 0, 180, 288, False),
    (32, 80, 112, 288, True), (32, 80, 111, 288, False),                            # copies and cache fit into what is free
])
def test_room_for_second_copies_counts_the_cache(weights, cache, free, total, room):
    assert room_for_copies(weights, cache, free, total) is room


@pytest.mark.parametrize("n,KV,H,hd,keys,slices", [
    (8, 4, 32, 64, 128, 4), (8, 4, 32, 64, 64, 4), (8, 4, 32, 64, 32, 1), (8, 4, 32, 64, 16, 1), (16, 1, 40, 32, 64, 4),
    (1, 1, 16, 128, 64, 2), (8, 1, 64, 64, 64, 2), (1, 1, 16, 128, 128, 4),      # long merges
    (8, 32, 32, 128, 64, 4), (9, 32, 32, 128, 64, 2),                             # more groups than CUs
])
def test_slices_of_short_contexts_in_float32(n, KV, H, hd, keys, slices):
    """One workgroup's four slices where they are the faster: not for a single tile of keys, nor for two where
    its merge is long or the groups are many."""
    assert K.attn_decode_slices(n, KV, H, hd, F32, keys) == slices


@pytest.mark.parametrize("n,KV,H,hd,keys,page,slices", [
    (64, 4, 32, 64, 2048, 20, 8), (64, 4, 32, 64, 2048, 24, 8), (72, 4, 32, 96, 8192, 20, 7), (20, 32, 32, 64, 4096, 12, 3),       # 32 columns: eight waves a CU
    (8, 32, 32, 128, 2048, 20, 4), (9, 32, 32, 128, 2048, 20, 7), (64, 4, 32, 64, 640, 20, 4), (32, 8, 256, 64, 640, 16, 8), (64, 4, 128, 64, 2048, 16, 8),
    (64, 4, 32, 64, 2048, 16, 4), (64, 4, 32, 64, 1 << 17, 48, 4), (14, 32, 32, 128, 16384, 16, 4), (16, 32, 32, 64, 8192, 32, 4),    # 16: whole last rounds
    (9, 32, 32, 64, 512, 16, 4), (9, 32, 32, 64, 1024, 16, 8), (9, 32, 32, 64, 4096, 16, 16), (12, 32, 32, 64, 1024, 16, 4), (12, 32, 32, 64, 2048, 16, 8), (12, 32, 32, 128, 8192, 16, 8),
    (17, 32, 32, 64, 8192, 16, 16), (72, 4, 32, 96, 4096, 16, 16), (72, 4, 32, 96, 2048, 16, 8), (28, 32, 32, 64, 2048, 16, 8), (100, 32, 32, 64, 8192, 16, 4)])
def test_slices_of_many_groups_in_float32(n, KV, H, hd, keys, page, slices):
    """From one group of heads per CU on: by the kernel that takes the pages, and on 16 columns by how full the last round of workgroups is."""
    assert K.attn_decode_slices(n, KV, H, hd, F32, keys, page) == slices


@pytest.mark.parametrize("n,heads,row,rank,keys,window,slices", [
    (8, 32, 576, 512, 1024, 0, 8), (8, 32, 576, 512, 4096, 0, 16), (33, 32, 576, 512, 4096, 0, 2), (33, 32, 288, 256, 4096, 0, 2), (33, 32, 704, 512, 4096, 0, 2),
    (33, 32, 192, 128, 4096, 0, 4), (33, 16, 72, 64, 4096, 0, 8), (16, 128, 400, 128, 4096, 0, 4), (33, 32, 424, 256, 4096, 0, 4), (33, 32, 384, 256, 4096, 0, 2),
    (4, 16, 72, 64, 300, 0, 4), (1, 16, 576, 512, 0, 100, 2), (64, 32, 576, 512, 4096, 0, 0)])
def test_slices_of_latent_attention_by_what_a_cu_holds(n, heads, row, rank, keys, window, slices):
    assert K.attn_latent_slices(n, heads, rank, BF16, window, keys, row) == slices


@pytest.mark.parametrize("kind,n,m,k,dtype,want", [
    (K.LINEAR_RESID, 64, 2048, 5632, torch.bfloat16, True), (K.LINEAR_SWIGLU, 64, 11264, 2048, torch.bfloat16, True),
    (K.LINEAR_ROPE, 64, 2560, 2048, torch.bfloat16, True), (K.LINEAR_RESID, 65, 2048, 5632, torch.bfloat16, False),
    (K.LINEAR_RESID, 16, 4096, 14336, torch.bfloat16, True), (K.LINEAR_RESID, 17, 4096, 14336, torch.bfloat16, False),
    (K.LINEAR_SWIGLU, 16, 28672, 4096, torch.bfloat16, True), (K.LINEAR_SWIGLU, 17, 28672, 4096, torch.bfloat16, False),
    (K.LINEAR_RESID, 8, 4112, 4096, torch.bfloat16, False), (K.LINEAR_RESID, 8, 2048, 2040, torch.bfloat16, False),
    (K.LINEAR_PARTS, 8, 2048, 2048, torch.float32, True), (K.LINEAR_PARTS, 17, 2048, 2048, torch.float32, False),
    (K.LINEAR_SWIGLU, 8, 131072, 4096, torch.float32, False)])
def test_products_without_staging_are_taken_by_size(kind, n, m, k, dtype, want):
    """256 CUs: up to 16 rows always, beyond while the busiest CU's rows stay below 380 KB; sums of squares for 4,096 columns at
    most, K in whole steps, float32 weights below 2 GiB (they are read without their copy too)."""
    assert K.linear_rows_best(kind, n, m, k, dtype) is want


def test_half_tiles_of_weights_only_where_half_the_cus_are_idle():
    assert K.linear_rows_parts(16, 2048, 2048) == 256 and K.linear_rows_parts(17, 2048, 2048) == 128
    assert K.linear_rows_parts(8, 2064, 2048) == 129 and K.linear_rows_parts(8, 2048, 2080) == 128
    assert K.linear_rows_parts(8, 4096, 4096) == 256 and K.linear_rows_parts(8, 4112, 4096) == 0


class _Recorder:
    """Stands for the context, the runtime and the norm of a product whose launch is only asked for."""

    def __init__(self, dtype, feeds=None, **options):
        self.runtime, self.options, self.dtype, self.feeds = self, options, dtype, feeds

    def buf(self, tag, shape, dtype):
        return torch.empty(shape, dtype=dtype)


@pytest.mark.parametrize("n,m,k,feeds,kernel", [
    (2, 2040, 2040, None, "gemv"), (3, 2040, 2040, None, "decode_batch"), (2, 4112, 4112, None, "decode_batch"),
    (2, 2048, 5632, (K.LINEAR_ROPE, 2560, 2048), "rows"), (2, 2040, 5632, (K.LINEAR_ROPE, 2856, 2040), "gemv"),
    (3, 2040, 5632, (K.LINEAR_ROPE, 2856, 2040), "rows"), (2, 2040, 5632, (K.LINEAR_SWIGLU, 11264, 2040), "rows"),
    (1, 2048, 2048, None, "gemv"), (5, 2040, 2040, None, "decode_batch"), (4, 1024, 1024, None, "rows"),
    (4, 1024, 2816, (K.LINEAR_ROPE, 1536, 1024), "rows"), (2, 1024, 2816, (K.LINEAR_ROPE, 1536, 1024), "rows")])
@pytest.mark.parametrize("copied", [True, False])
def test_few_rows_of_float32_leave_the_gemv_where_that_is_the_faster_way(n, m, k, feeds, kernel, copied, monkeypatch):
    """Two rows whose K is in no whole steps stay with the gemv unless the decode-batch kernel has a tile for every CU; so do those
    whose scaled rows the product behind the norm would not take.  Without the copy of the weights two rows leave it only where nothing
    is staged and K is beyond 1,024."""
    went = []
    if not copied and n == 2 and not (m == 2048 and feeds):
        kernel = "gemv"
    monkeypatch.setattr(K, "linear_resid", lambda *a, **b: went.append("gemv"))
    monkeypatch.setattr(K, "linear_rows", lambda *a, **b: went.append("rows"))
    monkeypatch.setattr(K, "fused_linear", lambda *a, **b: went.append("decode_batch"))
    rt = _Recorder(F32, feeds and (*feeds, copied))
    rt.weight = torch.empty(m)
    rt.eps = 1e-5
    x, w = torch.empty(n, k), torch.empty(m, k)
    normed = products.linear_into(rt, x, w, ResidualSink(torch.empty(n, m), rt), "t", object() if copied else None)
    if kernel == "gemv" and K.resid_parts(n, m, k, F32) == 0:       # (more columns than its sums of squares are read for)
        assert normed is None and not went
    else:
        assert went == [kernel] and (normed.xw is None) == (kernel == "gemv")
    assert products.decode_batch_fits(rt, x, m, copied) == (n > 2 or n == 2 and m >= 4096 and copied)


@pytest.mark.parametrize("lens,head_dim,want", [
    ([64], 128, True), ([63], 128, False), ([64] + [1] * 8, 128, True), ([64] + [1] * 9, 128, False), ([112] + [1] * 32, 128, True),
    ([111] + [1] * 32, 128, False), ([100] * 70, 128, True), ([480] + [1] * 200, 64, True), ([256] + [15] * 200, 64, False),
    ([64] + [1] * 200, 192, True), ([64] + [1] * 200, 129, True), ([64] + [1] * 200, 193, False), ([1] * 8, 192, False)])
def test_sixteen_tokens_at_a_time_only_where_short_spans_are_few(lens, head_dim, want):
    assert takes_sixteens(lens, head_dim) is want


@pytest.mark.parametrize("n,m,k,dtype,unary,want", [
    (1, 2048, 1024, BF16, False, False), (1, 2048, 1056, BF16, False, True), (6, 2048, 2048, BF16, False, True),
    (7, 2048, 2048, BF16, False, False), (7, 2048, 2080, BF16, False, True), (8, 2064, 2048, BF16, False, True), (8, 1024, 1056, BF16, True, False), (8, 4096, 1056, BF16, True, True), (8, 1024, 1024, BF16, True, False),
    (9, 2048, 2048, BF16, False, False), (16, 2048, 2048, BF16, True, False), (17, 2048, 160, BF16, False, True),
    (17, 2048, 128, BF16, False, False), (17, 2048, 128, BF16, True, True), (32, 2048, 2816, BF16, False, True),
    (33, 2048, 2080, BF16, False, False), (33, 2048, 2048, BF16, False, True), (64, 5632, 1024, BF16, True, True),
    (32, 12304, 512, BF16, True, False), (32, 12288, 512, BF16, True, True), (8, 16384, 4096, BF16, False, False),
    (5, 64, 64, F32, False, True), (6, 64, 64, F32, False, False), (8, 2816, 64, F32, False, True), (8, 64, 544, F32, False, True),
    (9, 2816, 2816, F32, False, False)])
def test_plain_sums_without_staging_by_size(n, m, k, dtype, unary, want):
    """The lines of the rule, both sides of each."""
    rt, w = _Recorder(dtype), torch.empty(m, k, dtype=dtype)
    assert products.parts_rows(rt, n, w, object(), unary) is want


@pytest.mark.parametrize("kind,n,m,tiles", [
    (K.LINEAR_SWIGLU, 64, 11264, 4), (K.LINEAR_SWIGLU, 64, 4096, 4), (K.LINEAR_ROPE, 64, 2560, 4), (K.LINEAR_ROPE, 64, 6144, 6),
    (K.LINEAR_RESID, 64, 2048, 2), (K.LINEAR_RESID, 33, 4096, 3), (K.LINEAR_PARTS, 48, 4112, 3), (K.LINEAR_PARTS, 48, 2048, 2)])
def test_rows_that_the_busiest_cu_reads(kind, n, m, tiles):
    """As the launch shares the tiles of columns and the halves of the rows out; beyond three tiles of columns a CU the products are not
    taken with more than 16 rows."""
    assert K.library().kllm_linear_rows_row_tiles(kind, n, m, 2048) == tiles
    assert K.linear_rows_best(K.LINEAR_SWIGLU, 17, 12288, 512) and not K.linear_rows_best(K.LINEAR_SWIGLU, 17, 12304, 512)
    assert K.linear_rows_best(K.LINEAR_SWIGLU, 16, 12304, 512)


@pytest.mark.parametrize("n,m,k,dtype,want", [(4, 2048, 2048, BF16, True), (5, 2048, 2048, BF16, False), (16, 512, 1024, BF16, False),
                                              (16, 2064, 2048, BF16, True), (16, 2048, 2080, BF16, True), (16, 2048, 2048, F32, True)])
def test_half_tiles_of_weights_want_rows_in_the_lanes_order(n, m, k, dtype, want):
    assert K.linear_rows_best(K.LINEAR_RESID, n, m, k, dtype, False) is want
    assert K.linear_rows_best(K.LINEAR_RESID, n, m, k, dtype, True)


@pytest.mark.parametrize("n,m,k,dtype,whole", [
    (64, 2560, 2048, BF16, False), (1024, 2560, 2048, BF16, False), (1280, 2560, 2048, BF16, True), (1800, 2560, 2048, BF16, True),
    (2048, 2560, 2048, BF16, True), (1024, 6144, 4096, BF16, False), (1280, 6144, 4096, BF16, True), (450, 12288, 4096, BF16, False),
    (700, 12288, 4096, BF16, True), (1800, 2560, 2048, F32, False), (1400, 2560, 2048, F32, True), (300, 2560, 1 << 23, BF16, False)])
def test_prompt_projections_in_one_slice(n, m, k, dtype, whole):
    """Rotation and append in the product's end wherever one slice is the fastest product, and in bfloat16 where the slices' way out and back costs
    more than they give."""
    assert K.gemm_rope_best(n, m, k, dtype) is whole
    assert products.prompt_rope(_Recorder(dtype), n, torch.empty(m, k, dtype=dtype, device="meta")) is whole


@pytest.mark.parametrize("kv_heads,head_dim,page_size,dtype,direct", [
    (4, 64, 64, F32, True), (32, 128, 65520, F32, True), (32, 128, 65536, F32, False), (32, 128, 131072, F32, False), (1, 32, 8388592, F32, True),
    (1, 32, 8388608, F32, False), (8, 128, 2048, BF16, True), (2047, 128, 2048, BF16, True), (2048, 128, 2048, BF16, False)])
def test_pages_whose_places_fit_31_bits(kv_heads, head_dim, page_size, dtype, direct):
    """Kernels that hold a place in a page in 31 bits get no page of 2 GiB and more."""
    assert K.attn_direct_pages(kv_heads, head_dim, page_size, dtype) is direct
    assert direct == (2 * kv_heads * head_dim * page_size * (4 if dtype == F32 else 2) < 2 ** 31)


@pytest.mark.parametrize("heads,head_dim,spans,window,shared", [
    (32, 64, [(0, 45)], 0, True), (32, 64, [(0, 700)], 0, True), (32, 64, [(0, 2048)], 256, True), (32, 64, [(0, 500)] * 4, 0, True),
    (32, 64, [(0, 40)] * 16, 0, False), (64, 64, [(0, 40)] * 16, 0, False), (32, 64, [(1000, 8)] * 24, 0, True),
    (40, 96, [(0, 6)] * 29, 1024, False), (32, 96, [(0, 40)] * 16, 0, False), (32, 96, [(0, 2048)], 256, False), (32, 96, [(0, 2048)], 0, True),
    (32, 128, [(0, 2048)], 256, False), (64, 128, [(300, 100)] * 8, 256, False), (64, 128, [(0, 2048)], 0, True), (40, 128, [(0, 51)] * 24, 0, False),
    (32, 128, [(0, 700)], 0, True), (8, 128, [(0, 18)] * 33, 64, False), (16, 32, [(0, 2048)], 0, True), (16, 32, [(0, 40)] * 16, 0, True)])
def test_float32_prompts_whose_keys_four_waves_share(heads, head_dim, spans, window, shared):
    """Many short chains of tiles go to the kernel with a wave to 32 tokens, as they did when it was the only one; unknown keys do not."""
    n_rows = sum(n for _, n in spans)
    keys = [min(a + min(t + 128, n), window + 128) if window else a + min(t + 128, n) for a, n in spans for t in range(0, n, 128)]
    assert K.attn_f32_prompt_shared(len(keys), heads, head_dim, n_rows, sum(keys), max(keys), window) is shared
    assert K.attn_f32_prompt_shared(len(keys), heads, head_dim, n_rows, 0, 0, window)


@pytest.mark.parametrize("heads,kv,head_dim,tokens,context,table,slices,blocks,total,longest,block_slices,window,at_least,at_most", [
    (32, 8, 128, 1, 4424, (70, 64), 32, 1, 45, 45, 4, 0, 8, 16), (12, 4, 128, 6, 4000, (63, 64), 21, 6, 1500, 479, 2, 0, 4, 11),
    (12, 4, 128, 4, 4088, (64, 64), 32, 2, 250, 184, 4, 0, 8, 16), (8, 2, 128, 16, 1492, (24, 64), 16, 2, 100, 75, 4, 1024, 4, 8),
    (32, 8, 64, 1, 3200, (50, 64), 32, 3, 300, 162, 1, 0, 2, 16), (64, 8, 128, 1, 6400, (101, 64), 64, 1, 13, 13, 4, 0, 8, 32),
    (32, 32, 128, 20, 560, (30, 64), 1, 4, 7000, 1920, 2, 0, 1, 1), (32, 8, 128, 20, 560, (30, 64), 4, 4, 7000, 1920, 2, 0, 1, 1),
    (32, 4, 64, 2, 100, (2, 64), 16, 1, 40, 40, 1, 0, 1, 1), (32, 32, 128, 2, 100, (2, 64), 8, 1, 40, 40, 4, 0, 1, 1),
    (8, 2, 128, 7, 9000, (600, 16), 16, 1, 24, 24, 4, 256, 1, 2), (12, 4, 128, 8, 17, (112, 16), 16, 3, 5000, 1790, 4, 0, 0, 0),
    (16, 16, 128, 27, 53, (35, 64), 1, 3, 6000, 2184, 4, 0, 0, 0)])
def test_workgroups_of_decode_tokens_beside_prompt_blocks(heads, kv, head_dim, tokens, context, table, slices, blocks, total, longest, block_slices,
                                                          window, at_least, at_most):
    """Long contexts beside a short portion are shared out, short ones and those behind a window are not, and blocks that are better off in slices get a
    launch of their own.  Without the contexts: by the table's width."""
    ask = lambda keys: K.attn_step_workgroups(head_dim, blocks, heads, kv, tokens, *table, slices, total, longest, keys, block_slices, window)
    assert at_least <= ask(context) <= at_most, ask(context)
    assert ask(0) == ask(table[0] * table[1])


def test_contexts_that_a_step_is_split_by():
    from kllm_amd.parts.attention import CausalSelfAttention as A
    part = A.__new__(A)
    part.window, part.chunk = 0, 0
    short = A.SHORT_SPAN
    assert part.step_values([0, 1, 301, 302], [1, 300, 1, short], [700, 100, 1500, 30]) == {
        "keys_total": 228 + 356 + 400, "keys_longest": 400, "keys_token": 1501}
    assert part.step_values([0], [200], [0])["keys_token"] == 0
    part.step_values_key = "k"
    ctx = types.SimpleNamespace(values={"k.keys_total": 5, "k.keys_longest": 4}, h_span_start=[0], h_span_len=[1], h_span_pos=[9])
    assert part._keys_read(ctx) == (5, 4, 0)                   # a part of its own that says the blocks' numbers only
    ctx.values = {}
    assert part._keys_read(ctx) == (0, 0, 10)
