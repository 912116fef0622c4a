"""Matrix products of the parts: choice of kernel and of a split of K.

``linear`` computes x . w^T for x [n, k] and w [m, k].  With a float32 result
it returns partial sums [nsplit, n, m] that the consuming kernel adds (norm,
rotary + append, SiLU gate); with the compute dtype as result it returns
[n, m].  Which kernel runs depends only on the dtype and on n (products with the step after
them in their launch, and ``decode_linear``, have the tiled copy of the weights and go to ``K.linear_rows``
first: up to 64 rows of bfloat16, 2 to 16 of float32, see ``K.linear_rows_best``):

  n <= 8    float32: gemv with X in LDS and the whole of K in one wave (no
            partial sums), if the sizes fit; bfloat16 up to 4 rows: the streaming
            gemv, K cut into slices for long rows (measured faster than the
            former for a plain product; the fused epilogues are another matter)
  float32   else: MFMA tiles with 32-bit operands (true 32-bit; K in slices for
            few rows, where one wave's chain of products bounds the time), or
            tiled FMA where K is no multiple of 4
  bfloat16  n <= 64: MFMA skinny (n <= 16 and one float32 result wanted: the
            decode-batch kernel with all of K in a workgroup; from 17 rows on: MFMA
            tiles of 64 rows)
            else: MFMA tiles (K in slices where the library's estimate of the product and of
            the kernel that adds the slices is the least with them),
            or the vendor library (torch.matmul) when the engine option
            ``gemm`` is "library" -- the reference uses its vendor library for
            every product (backend/model.cu:494-503)

Sizes that the MFMA kernels do not take (K not a multiple of 8) go to the plain
kernel.
"""

from __future__ import annotations

import functools

import torch

from .. import kernels as K

def _gemv_split(dtype, n, m, k):
    """Slices of K for the streaming gemv: a wave covers two rows and up to
    2048 (bfloat16) or 1024 (float32) of K with all loads in flight; K is cut
    unless the rows alone already give the chip enough waves."""
    per = 2048 if dtype == torch.bfloat16 else 1024
    if m // 2 >= 4096:
        return 1
    return int(max(1, min(16, -(-k // per))))


def _skinny_split(n, m, k):
    """Slices of K for the skinny MFMA kernel: at most 512 of K per workgroup
    (its LDS stage); more slices while the chip has no workgroup per CU and a
    slice keeps 128 of K.  Idle CUs cost more than the partial sums that a
    further slice writes (measured up to 64 rows)."""
    nsplit = -(-k // 512)
    wgs = -(-m // 64)
    while wgs * nsplit < K.device_cus() and k // (nsplit * 2) >= 128:
        nsplit *= 2
    return _no_empty_slice(nsplit, k, 32)


# K of a stage of the MFMA tiles, 128 bytes.  Their slices are rounded up to two stages, or to one where two
# would leave the last slice empty.
_STAGE_BF16, _STAGE_F32 = 64, 32


def _no_empty_slice(nsplit, k, unit):
    """The most slices up to ``nsplit`` of which none is empty, where a kernel rounds a slice of K up
    to ``unit``."""
    nsplit = int(nsplit)
    while nsplit > 1 and (-(-(-(-k // nsplit)) // unit) * unit) * (nsplit - 1) >= k:
        nsplit -= 1
    return nsplit


def _mfma_f32_split(n, m, k):
    """Slices of K for the float32 MFMA kernel.  Up to 64 rows (one row of tiles of 64 x 128) a wave's
    own chain of products bounds the time, so a CU should have two tiles side by side: up to 16 slices of
    at least 128 of K (2,048 x 5,632 at 64 rows, in us with the sum of the slices: 32 with 8, 26 with 11, 24 with 16; 4,096 x
    14,336 75 with 8, 70 with 16)."""
    if n > 64:
        return K.gemm_prompt_slices(n, m, k, torch.float32)
    tiles = -(-m // 128)
    nsplit = max(1, min(16, k // 128, -(-2 * K.device_cus() // tiles)))
    return _no_empty_slice(nsplit, k, _STAGE_F32)


def _tiles_beat_skinny(n, m, k):
    """Decode batches of more than 16 rows (two or more of the skinny kernel's 16-row
    tiles): the tiled kernel (tiles of 64 rows, both operands through LDS in whole cache lines) takes nearly
    the same time from 20 to 64 rows, the time of its weights; the skinny one, whose
    workgroups each stage all rows of X for 512 of K and leave up to 28 partial sums, grows
    with the rows.  Measured, tiled against skinny in us, at 64 rows: 2,048 x 5,632: 10.7 / 13.5;
    2,560 x 2,048: 6.8 / 8.6; 2,048 x 2,048: 6.2 / 6.9; 11,264 x 2,048: 14.1 / 19.7; 4,096 x 4,096:
    10.4 / 15.1; 4,096 x 14,336: 23.9 / 41.1; 28,672 x 4,096: 52.5 with the gate / 72.7.  At 20 rows:
    9.5 / 9.4; 5.6 / 6.4; 5.2 / 5.4; 11.2 / 13.4; 8.8 / 10.6; 22.2 / 30.0."""
    return n > 16


def _decode_tile_split(n, m, k):
    """Slices of K for a decode batch on the tiled kernel (one row of tiles of 64).  Below 40 M weights: slices of
    at least 256 of K until every second CU has a tile of 128 columns, then
    further ones of at least 512, up to 16 (at 64 rows, in us by slices, alone in a graph / with the sums added: 2,048 x 5,632:
    13.0 / 14.9 with 4, 9.4 / 11.5 with 8; 2,048 x 2,048: 7.1 / 8.9 with 4, 5.8 / 7.6 with 8; 4,096 x 4,096: 11.3 / 13.8 with 4, 10.1 /
    13.2 with 8, 11.4 / 15.5 with 16; 11,264 x 2,048, which gets four: 12.0 / 15.7 with 2, 13.2 / 17.3 with 4, 14.0 / 19.2 with 8;
    at 17 rows 11.1 / 13.2, 10.6 / 13.0 and 10.8 / 13.5).  Where that stops between two powers and the tiles of 128
    columns leave CUs idle: as many slices of 512 as there are (2,048 x 5,632 with the norm that adds
    the slices, 8 / 11 / 15: 17 rows 14.3 / 13.5 / 13.3, 32 rows 14.7 / 14.1 / 14.3, 48 rows 15.5 / 15.0 /
    15.1; the sums of more slices cost more with every row: 8 / 11 with the sums added, 48 rows 10.8 / 9.8, 56 11.1 / 10.5, 64
    11.5 / 11.0).  Larger weights: up to 8 slices
    of at least 512 of K towards two workgroups a CU, four where K is deep (12,288 x 4,096: 26.2
    with 2, 22.3 with 4, 24.6 with 8; 4,096 x 14,336: 34.4 with 4, 23.9 with 8)."""
    cus, nsplit = K.device_cus(), 1
    if m * k < 40_000_000:
        tiles = -(-m // 64)
        while nsplit < 16 and ((tiles * nsplit < cus and k // (2 * nsplit) >= 256) or k // (2 * nsplit) >= 512):
            nsplit *= 2
        if n <= 48 and nsplit < k // 512 <= 16 and -(-m // 128) * (k // 512) <= cus:
            nsplit = k // 512
    else:
        tiles = -(-m // 128)
        reach = (4 if k >= 8192 and tiles <= cus else 2) * cus
        while nsplit * 2 <= min(8, reach // tiles, k // 512):
            nsplit *= 2
    return _no_empty_slice(nsplit, k, _STAGE_BF16)


def choose(dtype, n, m, k, options=None):
    """(algorithm, nsplit) for a product of these sizes."""
    options = options or {}
    forced = options.get("gemm_algo")
    if forced is not None:
        return forced, 1
    if dtype == torch.float32 and K.gemv_fits(n, m, k, dtype) and not options.get("no_fused_gemv"):
        return K.GEMM_GEMV_LDS, 1
    if n <= 4 or (n <= 8 and dtype == torch.float32):
        return K.GEMM_GEMV, _gemv_split(dtype, n, m, k)
    if dtype == torch.float32:
        if k % 4 == 0 and not options.get("no_mfma_f32"):
            return K.GEMM_MFMA_F32, _mfma_f32_split(n, m, k)
        return K.GEMM_TILED_F32, 1
    if k % 8 != 0:
        return (K.GEMM_GEMV, 1) if n <= 8 else (K.GEMM_PLAIN, 1)
    if n <= 64:
        if _tiles_beat_skinny(n, m, k) and options.get("gemm") != "library":
            return K.GEMM_MFMA_BF16, _decode_tile_split(n, m, k)
        return K.GEMM_SKINNY_BF16, _skinny_split(n, m, k)
    if options.get("gemm") == "library":
        return "library", 1
    return K.GEMM_MFMA_BF16, K.gemm_prompt_slices(n, m, k)


@functools.lru_cache(maxsize=4096)
def _resid_tiles(n, m, k, dtype=torch.bfloat16):
    """(tiles per workgroup, partial sums of squares per row) of a decode batch's residual
    product: as few tiles to a workgroup as keep the sums of squares within what the
    consumer reads (one tile where the rows go through LDS in passes over K); (1, 0) if the
    kernel does not take the sizes."""
    passes = K.fused_linear_passes(n, k, 1, dtype)
    if passes == 0 or (passes > 1 and (passes > K.FUSED_LINEAR_BEST_PASSES or n > K.FUSED_LINEAR_PASSES_BEST_ROWS)):
        return 1, 0
    tpw = 1
    while K.fused_resid_parts(n, m, k, tpw, dtype) == 0 and tpw < 64 and passes == 1:
        tpw *= 2
    return tpw, K.fused_resid_parts(n, m, k, tpw, dtype)


def tiled_copy(runtime, w, kind, rope=None):
    """A second copy of a weight matrix in the order the decode-batch kernel's lanes read it
    (``K.fused_linear_tile``), or None where that kernel does not run: other dtypes, sizes it
    does not take, or ``EngineOptions.extra["no_tiled_weights"]`` (the copies double the
    memory of the weights they are made of; decode batches of 2 to 16 tokens stream them 20 to
    30 % faster than the row-major matrix).  float32: only where the engine found room for all of them behind
    its cache (``Runtime.second_copies``); without them 2 / 4 / 8 tokens at 1.1B sizes take 1,494 / 1,495 / 1,562 us a step, with
    them 1,404 / 1,434 / 1,534, and the sums are the same."""
    if (w is None or not w.is_cuda or w.shape[1] % (4 if w.dtype == torch.float32 else 8)
            or runtime.options.get("no_tiled_weights") or runtime.options.get("no_fused_linear")):
        return None
    if w.dtype == torch.float32 and (runtime.options.get("no_mfma_f32") or not runtime.second_copies):
        return None
    return K.fused_linear_tile(w, kind, rope)


def fused_f32(rt, n, m=None, k=None, copied=True):
    """Whether a float32 decode batch of n tokens runs on the matrix cores, with the step after a product in its launch
    (``K.linear_rows``, or the decode-batch kernel for sizes that one does not take: ``m``, the product's columns).  One row stays with the
    gemv, which has the same epilogues
    and the row in registers (a step in us, gemv against the matrix cores, of 1 / 2 / 4 tokens at 1.1B sizes: 1,436 / 1,516 / 1,708
    against 1,381 / 1,404 / 1,434, without room for the copies of the weights 2 / 4 tokens 1,535 / 1,723 against 1,494 / 1,495; at 8B
    sizes 6,103 / 6,262 / 6,610 against 6,392 / 6,166 / 6,197).  Its work per weight grows with the rows and the matrix cores' does
    not, and from nine on K went in slices whose sums other kernels added (16 at 8B sizes: 14.6 ms against 9.7 on the
    decode-batch kernel; 12: 9.1 there, 7.0 now).  The decode-batch kernel stages all rows first: two rows stay with the gemv, too, where it
    has fewer tiles than there are CUs (a step, gemv / decode-batch kernel, 2 / 3 / 4 tokens: width 2,040 x 8 layers 716 / 884 / 896 us against
    735 / 836 / 850; width 4,112 x 4 layers 896 / 912 / 929 against 864 / 850 / 898).  Without the copy of the weights (not
    ``copied``) two rows leave the gemv, which reads the weights in whole rows, only for ``K.linear_rows`` with ``k`` beyond 1,024 (a product alone
    1,024 x 1,024 3.9 / 4.9 us; a step of 2 tokens, layers of 1,024 columns, 692 / 739, of 2,048 839 / 797; of 5,120, whose residual products
    went to the decode-batch kernel, 1,173 / 1,264)."""
    opts = rt.options
    return (2 <= n <= 16 and (n > 2 or ((copied or k is None or k > 1024) if m is None else copied and m >= 16 * K.device_cus()))
            and not opts.get("no_fused_linear") and not opts.get("no_mfma_f32") and opts.get("gemm_algo") is None)


def _rows_options(rt, n, k, f32, w_tiled):
    """Whether the engine's options and the copy of the weights leave n rows of k to ``K.linear_rows``."""
    if f32:
        return fused_f32(rt, n, None, k, w_tiled is not None)
    opts = rt.options
    return (w_tiled is not None and opts.get("gemm") != "library" and not opts.get("no_fused_linear")
            and opts.get("gemm_algo") is None)


def rows_kernel(rt, kind, n, w, w_tiled, tiled_x):
    """Whether a product of n rows (``TiledRows``: ``tiled_x``) with the step after it runs on ``K.linear_rows``."""
    if n > K.LINEAR_ROWS_MAX:
        return False
    dtype, (m, k) = w.dtype, w.shape
    return K.linear_rows_best(kind, n, m, k, dtype, tiled_x) and _rows_options(rt, n, k, dtype == torch.float32, w_tiled)


def _sink_fits(rt, sink, n, m):
    opts, norm = rt.options, sink.norm
    return not (opts.get("no_fused_norm") or opts.get("gemm_algo") is not None or opts.get("no_fused_gemv")
                or tuple(sink.x.shape) != (n, m) or norm.weight is None or norm.weight.numel() != m)


def _feeds_rows(norm, n):
    """Whether the product behind ``norm`` runs on ``K.linear_rows`` and reads ``TiledRows``."""
    feeds = getattr(norm, "feeds", None)
    return feeds is not None and norm.runtime.dtype == torch.bfloat16 and K.linear_rows_best(feeds[0], n, feeds[1], feeds[2])


def _feeds_f32(rt, norm, n):
    """Whether the float32 product behind ``norm`` has a use for scaled rows: not where it stays with the gemv, which makes its rows'
    norm itself."""
    feeds = getattr(norm, "feeds", None)
    if feeds is None:
        return True
    kind, m, k, copied = feeds
    return fused_f32(rt, n, None if K.linear_rows_best(kind, n, m, k, torch.float32) else m, k, copied)


def _resid_rows(rt, norm, n, w, w_tiled, tiled_x):
    """Whether a residual product runs on ``K.linear_rows``: beyond 16 rows only where the next product does, too (a step of 32
    tokens at 8B sizes, whose gate product does not, 4,234 us without and 4,370 with the output projection here)."""
    if not rows_kernel(rt, K.LINEAR_RESID, n, w, w_tiled, tiled_x):
        return False
    return n <= 16 or _feeds_rows(norm, n)


def sink_takes_rows(rt, sink, n, w, w_tiled):
    """Whether ``linear_into`` will run the product of ``TiledRows`` on ``K.linear_rows``."""
    return sink is not None and n <= K.LINEAR_ROWS_MAX and w.dtype == torch.bfloat16 and _sink_fits(rt, sink, n, w.shape[0]) and _resid_rows(rt, sink.norm, n, w, w_tiled, True)


def linear_into(ctx, x, w, sink, tag, w_tiled=None):
    """x . w^T added to the residual stream of ``sink`` in the product's own
    epilogue: returns the ``Normed`` that stands for the norm behind the addition, or None
    if no kernel with that epilogue takes these sizes (the caller then returns the product
    and the norm adds it).  Up to four tokens on the gemv, whose consumer normalises the
    float32 rows as it stages them (4 % of a step of one token at width 2048); decode batches on
    the matrix cores, whose consumer scales its sums by the row instead."""
    from .base import Normed
    n, k = x.shape
    m = w.shape[0]
    rt = ctx.runtime
    rows = isinstance(x, K.TiledRows)            # (``sink_takes_rows`` said so)
    if not rows and not _sink_fits(rt, sink, n, m):
        return None
    norm = sink.norm
    f32 = x.dtype == torch.float32
    rows = rows or ((not f32 or _feeds_f32(rt, norm, n)) and _resid_rows(rt, norm, n, w, w_tiled, False))
    fused = f32 and (rows or fused_f32(rt, n, m, k, w_tiled is not None) and _feeds_f32(rt, norm, n))
    parts = 0 if fused else K.resid_parts(n, m, k, x.dtype)
    if parts:
        ss = ctx.buf(tag + ".ss", (n, -(-parts // 4) * 4), torch.float32)
        K.linear_resid(x, w, sink.x, ss)
        return Normed(sink.x, ss, parts, norm)
    if rows:
        parts = K.linear_rows_parts(n, m, k)
        stride = -(-parts // 4) * 4          # (room for eight columns to a sum whatever n is: a smaller step must not ask for more)
        ctx.buf(tag + ".ss", (n * max(stride, -(-m // 32) * 4),), torch.float32)
        ss = ctx.buf(tag + ".ss", (n, stride), torch.float32)
        if _feeds_rows(norm, n):
            xw = K.TiledRows(ctx.buf(tag + ".xw", (K.TiledRows.stored(n), m), x.dtype), n)     # for the product behind the norm
        else:
            xw = ctx.buf(tag + ".xw", (n, m), x.dtype)
        K.linear_rows(w_tiled or w, xw, K.LINEAR_RESID, x, resid=sink.x, norm_weight=norm.weight, ss_out=ss)
        return Normed(sink.x, ss, parts, norm, xw=xw)
    if not (fused if f32 else n <= K.FUSED_NORM_BEST_ROWS) or rt.options.get("no_fused_linear"):
        return None
    # a decode batch on the matrix cores: all of K in a workgroup, the addition in the epilogue, and
    # beside the stream its rows times the norm's weight in the compute dtype for a consumer that scales its sums
    tpw, parts = _resid_tiles(n, m, k, x.dtype)
    if parts == 0:
        return None
    ss = ctx.buf(tag + ".ss", (n, -(-parts // 4) * 4), torch.float32)
    xw = ctx.buf(tag + ".xw", (n, m), x.dtype)
    K.fused_linear(w_tiled if w_tiled is not None else w, xw, K.LINEAR_RESID, x=x, tiles_per_wg=tpw, resid=sink.x,
                   norm_weight=norm.weight, ss_out=ss)
    return Normed(sink.x, ss, parts, norm, xw=xw)


def prompt_rope(rt, n, w):
    """Whether a prompt's input projections (more than 64 rows) run on the MFMA tiles with all of K in one slice, where the rotation and
    the append are the end of a tile (``K.gemm_rope``)."""
    return (n > 64 and choose(w.dtype, n, *w.shape, rt.options)[0] in (K.GEMM_MFMA_BF16, K.GEMM_MFMA_F32)
            and (rt.options.get("gemm_algo") is not None or K.gemm_rope_best(n, *w.shape, w.dtype)))


def linear(ctx, x, w, tag, out_dtype=torch.float32, split=True, w_tiled=None):
    """x [n, k] . w [m, k]^T.  With a float32 result and ``split``: partial
    sums [nsplit, n, m] for a consumer that adds them; otherwise one [n, m]
    tensor of ``out_dtype``.  ``w_tiled``: the tiled copy of w (``tiled_copy`` with
    LINEAR_PARTS), taken where the decode-batch kernel runs."""
    n, k = x.shape
    m = w.shape[0]
    rt = ctx.runtime
    algo, nsplit = choose(x.dtype, n, m, k, rt.options)
    whole = not split or out_dtype != torch.float32
    if ((algo == K.GEMM_SKINNY_BF16 or (algo == K.GEMM_MFMA_F32 and fused_f32(rt, n))) and whole
            and out_dtype == torch.float32 and n <= 16 and K.fused_linear_fits(n, k, 1, x.dtype)
            and not rt.options.get("no_fused_linear")):
        # one float32 result from a decode batch (the logits): all of K in one workgroup, so
        # that no partial sums have to be added afterwards
        y = ctx.buf(tag, (1, n, m), torch.float32)
        K.fused_linear(w_tiled if w_tiled is not None else w, y, K.LINEAR_PARTS, x=x, tiles_per_wg=4 if m >= 16384 else 1)
        return y[0]
    if algo == "library":
        K.bypass_recorded()             # the library is called through torch: behind what was recorded
        if out_dtype == torch.float32:
            # float32 sums straight from the library's accumulators: a result that the caller
            # wants in 32-bit (a residual delta, logits) is never rounded to bfloat16 on the way
            y32 = ctx.buf(tag + ".f32", (1, n, m), torch.float32)
            torch.mm(x, w.t(), out_dtype=torch.float32, out=y32[0])
            return y32[0] if whole else y32
        y = ctx.buf(tag, (n, m), x.dtype)
        torch.matmul(x, w.t(), out=y)
        return y
    if (algo == K.GEMM_MFMA_BF16 or algo == K.GEMM_PLAIN
            or (algo == K.GEMM_MFMA_F32 and (nsplit == 1 or not whole))):   # write either dtype themselves
        if whole:
            y = ctx.buf(tag, (n, m), out_dtype)
            K.gemm(x, w, y, algo, 1)
            return y
        y = ctx.buf(tag, (nsplit, n, m), torch.float32)
        K.gemm(x, w, y, algo, nsplit)
        return y
    parts = ctx.buf(tag, (nsplit, n, m), torch.float32)       # float32 partial sums only
    K.gemm(x, w, parts, algo, nsplit)
    if not whole:
        return parts
    if nsplit == 1 and out_dtype == torch.float32:
        return parts[0]
    y = ctx.buf(tag + ".sum", (n, m), out_dtype)
    K.sum_splits(parts, y)
    return y


def decode_batch_fits(rt, x, m, copied=True):
    """Whether a product of these rows with m columns runs on the decode-batch kernel (up to 16 rows, all of K
    in a workgroup; float32 see ``fused_f32``)."""
    n, k = x.shape
    if x.dtype == torch.float32 and not fused_f32(rt, n, m, k, copied):
        return False
    return n <= 16 and K.fused_linear_fits(n, k, 1, x.dtype)


@functools.lru_cache(maxsize=4096)
def _parts_best(n, m, k, dtype, unary, copied=True):
    """Whether ``K.linear_rows`` is the fastest way to plain sums, or (``unary``) an activation of them, of n rows that are read row by row.
    For bfloat16 up to 16 rows this asks where it beats the kernels other than the decode-batch kernel: what that one would run, ``_unstaged`` sends to
    ``K.linear_rows`` as well, so that the lines for those rows matter only where K is too long for its passes.  They, their figures below and the float32 lines
    were measured before ``K.linear_rows`` asked for the weights first; its times are up to 1.5 us a product shorter now.
    The decode-batch kernel has the rows in LDS, this one reads up to sixteen of them a load: up to eight rows it is the faster one where
    K is long enough, of 9 to 16 not (a step of Nusilix layers of 1,024 columns, there / here, with K of 1,024 here, too: 1 token 601 / 608 us, 2
    606 / 617, 8 678 / 714; us a product: 8 rows 2,048 x 1,024 3.8 / 4.6, 2,048 x 4,096 6.8 / 6.2, 1,024 x 1,408 in a step 3.9 / 5.3, 2,048 x 2,048 4.9 /
    5.2; a step at Natenex sizes, 16 rows 898 / 903).  Beyond 16 rows it takes the place of K in slices from the tiles, which the consumer adds, and
    of an activation's launch (a step at Natenex sizes, without and with: 24 tokens 1,123 / 894, 48 1,268 / 1,192, 64 1,538 / 1,524, a
    prompt of 20 1,004 / 761, of 60 1,146 / 1,131), but for sums of little K and, beyond 32 rows, of long K (a product and a
    kernel that adds the slices, there / here: 48 rows 1,024 x 64 6.1 / 7.6, 1,024 x 2,816 8.9 / 12.3), nor for more than three
    tiles of columns a CU (32 rows 14,336 x 1,024 with the activation 12.3 / 18.7)."""
    if m >= 16384 or not K.linear_rows_best(K.LINEAR_PARTS, n, m, k, dtype, False):
        return False
    if dtype == torch.float32:
        if not copied and (n == 2 and k <= 2048 or n > 5 and k <= 1024):
            return False          # (without the copy: a step of 8 tokens of Nusilix layers of 1,024 columns 970 us there, 987 here)
        return n <= 5 or n <= 8 and (k > 512 or m > 2048)      # (8 rows, 2,048 x 512: 4.5 us there, 4.8 here; 2,816 x 512 5.2 / 5.0)
    if n <= 8:
        return k > 1024 and (n <= 6 or k > 2048 or m > 2048)
    if n <= 16 or m > 48 * K.device_cus():
        return False
    return unary or (k > 128 and (n <= 32 or k <= 2048))


def parts_rows(rt, n, w, w_tiled, unary=False):
    """Whether ``decode_linear`` runs on ``K.linear_rows`` (``_parts_best``)."""
    if n > K.LINEAR_ROWS_MAX:
        return False
    dtype, (m, k) = w.dtype, w.shape
    return _parts_best(n if n <= 8 else -(-n // 16) * 16, m, k, dtype, unary, w_tiled is not None) and _rows_options(rt, n, k, dtype == torch.float32, w_tiled)


def _unstaged(rt, n, m, k, dtype, w_tiled):
    """Whether plain sums, or an activation of them, of up to 16 rows of bfloat16 that ``_parts_best`` leaves to the decode-batch
    kernel come from ``K.linear_rows`` all the same.  That rule's figures are from before this kernel asked for the weights first and had its
    arguments with the launch; now it is the faster at every size tried (us a product, decode-batch kernel / this one, at 1, 8 and 16 rows:
    512 x 64 3.1 / 2.0, 3.4 / 2.4, 3.7 / 3.3; 1,024 x 512 3.4 / 2.4, 3.6 / 3.0, 3.9 / 3.8; 1,024 x 1,408 4.1 / 2.9, 4.4 / 3.4, 4.9 / 4.2; 2,048 x
    2,048 4.5 / 3.5, 4.9 / 3.9, 5.5 / 4.7; 4,096 x 512 3.6 / 3.3, 3.9 / 3.6, 4.2 / 4.2; 8,192 x 1,024 5.6 / 5.3, 6.2 / 5.6, 6.5 / 6.1; 2,048 x 5,632 9.2 /
    6.1, 8.9 / 7.4, 11.0 / 10.0; with an activation the same; steps: Natenex sizes 8 tokens 643 / 632, 16 tokens 800 / 770, Puladra layers of 1,024
    columns 1 token 1,063 / 969, Nusilix layers of 2,048 columns 12 tokens 518 / 495).  From 16,384 columns on and where K is no multiple of 32
    the decode-batch kernel stays."""
    return (dtype == torch.bfloat16 and w_tiled is not None and n <= 16 and k % 32 == 0 and m < 16384
            and _rows_options(rt, n, k, False, w_tiled))


def decode_linear(ctx, x, w, tag, w_tiled=None, unary=None):
    """``linear`` for a consumer that takes float32 sums either whole or in slices: ``K.linear_rows`` where it is the
    faster (``parts_rows``, ``_unstaged``); else decode
    batches of up to 16 rows run on the decode-batch kernel with all of K in a workgroup (one
    result, from the tiled copy of w where there is one); everything else as ``linear`` cuts it.
    ``unary`` = (activation without a gate, its constants): only where ``decode_batch_fits`` or ``parts_rows``;
    the result is then the activation of the sums in the compute dtype."""
    n, m = x.shape[0], w.shape[0]
    rt = ctx.runtime
    if parts_rows(rt, n, w, w_tiled, unary is not None):
        y = ctx.buf(tag, (n, m) if unary is not None else (1, n, m), x.dtype if unary is not None else torch.float32)
        K.linear_rows(w_tiled or w, y, K.LINEAR_PARTS, x, unary=unary)
        return y if unary is not None else y[0]
    if decode_batch_fits(rt, x, m, w_tiled is not None) and not rt.options.get("no_fused_linear") and rt.options.get("gemm_algo") is None:
        y = ctx.buf(tag, (n, m) if unary is not None else (1, n, m), x.dtype if unary is not None else torch.float32)
        if _unstaged(rt, n, m, w.shape[1], x.dtype, w_tiled):
            K.linear_rows(w_tiled, y, K.LINEAR_PARTS, x, unary=unary)
        else:
            K.fused_linear(w_tiled if w_tiled is not None else w, y, K.LINEAR_PARTS, x=x, tiles_per_wg=4 if m >= 16384 else 1, unary=unary)
        return y if unary is not None else y[0]
    if unary is not None:
        raise ValueError("decode_linear: the activation goes with the decode-batch kernel only")
    return linear(ctx, x, w, tag)
