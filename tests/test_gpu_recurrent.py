"""The recurrent kernels alone against their recurrences in double on the CPU, at the sizes where
their blocks, tiles and segments begin and end: spans of several requests side by side, some of
which continue from a state.

Bounds: every output is a sum of products in 32 bits along a chain that the decays shorten; with
unit inputs the difference from double stays within a few hundred roundings of 2^-24, 4e-5 relative
to the largest output."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64


def K():
    from kllm_amd import kernels
    return kernels


def spans_of(lens, fresh):
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    i32 = dict(dtype=torch.int32, device=DEV)
    token = torch.tensor([i for i, n in enumerate(lens) for _ in range(n)], **i32)
    pos = torch.tensor([0 if f else 7 for f in fresh], **i32)
    slots = torch.tensor([len(lens) - i for i in range(len(lens))], **i32)      # not in order, one unused
    return start, token, torch.tensor(start, **i32), pos, slots


def close(got, want, rel=4e-5):
    err = float((got.double().cpu() - want).abs().max())
    assert err <= rel * float(want.abs().max().clamp_min(1.0)), err


@pytest.mark.parametrize("dk,dv", [(8, 24), (64, 16), (65, 17), (128, 40), (136, 16), (200, 8), (256, 33)])
@pytest.mark.parametrize("lens,fresh", [([1, 1, 1], [0, 1, 0]), ([3, 16, 17], [1, 0, 1]), ([5, 33], [0, 1])])
@pytest.mark.parametrize("per_channel", [False, True])
def test_delta_scan(dk, dv, lens, fresh, per_channel):
    g = torch.Generator().manual_seed(dk + dv)
    n, H, G = sum(lens), 4, 2
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    k, q = (unit(torch.randn(n, G, dk, generator=g, dtype=F64)) for _ in range(2))
    v = torch.randn(n, H, dv, generator=g, dtype=F64)
    beta = torch.rand(n, H, generator=g, dtype=F64)
    decay = torch.rand(n, H, dk if per_channel else 1, generator=g, dtype=F64) ** 0.25
    decay[-1, 0] = 0.0                                                     # forgets everything
    state = torch.randn(len(lens) + 1, 5 + H * dk * dv, generator=g, dtype=F64)
    start, _, span_start, span_pos, slots = spans_of(lens, fresh)
    f = lambda t: t.float().to(DEV).contiguous()
    dev_state, out = f(state), torch.full((n, H * dv), float("nan"), device=DEV)
    gb = torch.stack([torch.ones(n, H) if per_channel else decay[..., 0], beta], dim=1)
    K().gated_delta_scan(f(q).view(n, -1), f(k).view(n, -1), f(v).view(n, -1), f(gb), out, dev_state, 5, slots, span_start,
                         span_pos, len(lens), H, G, dk, dv, f(decay).view(n, -1) if per_channel else None)
    state = state.float().double()
    k, q, v, beta, decay = (t.float().double() for t in (k, q, v, beta, decay))
    want = torch.zeros(n, H, dv, dtype=F64)
    for s in range(len(lens)):
        slot = int(slots[s])
        S = state[slot, 5:].view(H, dk, dv).clone() * (0.0 if fresh[s] else 1.0)
        for t in range(start[s], start[s + 1]):
            kk, qq = k[t].repeat_interleave(H // G, 0), q[t].repeat_interleave(H // G, 0)
            S = S * decay[t][:, :, None]
            u = beta[t][:, None] * (v[t] - (S * kk[:, :, None]).sum(1))
            S = S + kk[:, :, None] * u[:, None, :]
            want[t] = (S * qq[:, :, None]).sum(1)
        state[slot, 5:] = S.reshape(-1)
    close(out.view(n, H, dv), want)
    close(dev_state, state)


@pytest.mark.parametrize("blocks,bs", [(3, 8), (2, 40), (1, 130), (2, 256), (1, 1040)])
@pytest.mark.parametrize("lens", [[1], [1, 1, 1, 1, 1], [9, 1, 7], [40, 24], [64, 1], [3, 120, 2]])
@pytest.mark.parametrize("taps", [1, 2, 4, 5])
def test_recurrence_gates(blocks, bs, lens, taps):
    """Convolution, gates' products and decays: one tile of tokens and several, requests that meet
    within a tile and within a thread's run of tokens, blocks of odd sizes and of more inputs than LDS takes."""
    check_recurrence_gates(blocks, bs, lens, taps)


@pytest.mark.parametrize("blocks,bs,lens", [(2, 256, [300, 1, 99]), (2, 136, [33] * 30), (1, 1040, [1, 200, 100]),      # one tile of tokens, eight waves
                                            (8, 136, [1000, 1, 1, 45]), (33, 8, [500, 1, 13])])                  # two tiles
@pytest.mark.parametrize("taps", [1, 4, 8, 9])
def test_recurrence_gates_of_prompts(blocks, bs, lens, taps):
    """The same where the tokens and blocks give the chip workgroups enough for the wider forms."""
    check_recurrence_gates(blocks, bs, lens, taps)


def check_recurrence_gates(blocks, bs, lens, taps):
    g = torch.Generator().manual_seed(bs + taps)
    n, W, fresh = sum(lens), blocks * bs, [i % 2 for i in range(len(lens))]
    r = lambda *s: torch.randn(*s, generator=g)
    proj, x_bias, conv_w, conv_b = r(2, n, 2 * W), r(W), r(W, taps) * 0.5, r(W) * 0.3
    wr, wi, br, bi = r(blocks, bs, bs) / bs ** 0.5, r(blocks, bs, bs) / bs ** 0.5, r(W) * 0.3, r(W) * 0.3
    rate = torch.rand(W, generator=g)
    state = r(len(lens) + 1, 3 + W * (taps - 1))
    start, token, span_start, span_pos, slots = spans_of(lens, fresh)
    d = lambda t: t.to(DEV).contiguous()
    a, b = (torch.full((n, W), float("nan"), device=DEV) for _ in range(2))
    K().linear_recurrence_prep(d(proj), d(x_bias), d(conv_w), d(conv_b), taps, d(state), 3, d(wr), d(wi), d(br), d(bi),
                               d(rate), token, slots, span_start, span_pos, a, b, blocks)
    x = proj.double().sum(0)[:, W:] + x_bias.double()
    u = torch.zeros(n, W, dtype=F64)
    for s in range(len(lens)):
        before = state[int(slots[s]), 3:].view(W, taps - 1).double().t() * (0.0 if fresh[s] else 1.0)
        rows = torch.cat([before, x[start[s]:start[s + 1]]])
        for j in range(taps):
            u[start[s]:start[s + 1]] += rows[j:j + lens[s]] * conv_w[:, j].double()
    u = u + conv_b.double()
    ub = u.view(n, blocks, bs)
    gate = lambda w, bias: torch.sigmoid(torch.einsum("nbi,bio->nbo", ub, w.double()).reshape(n, W) + bias.double())
    log_a = -rate.double() * gate(wr, br)
    close(a, torch.exp(log_a))
    close(b, torch.sqrt(-torch.expm1(2 * log_a)) * gate(wi, bi) * u, rel=1e-4)   # (the root of a small difference)


@pytest.mark.parametrize("n", [8, 100, 400, 1200])
@pytest.mark.parametrize("blocks,bs", [(4, 256), (1, 1040)])
def test_recurrence_gates_add_in_short_chains(n, blocks, bs):
    """How far a gate's sums are from 64 bits, read off the added term: with an input gate far below zero, sigmoid(z) =
    exp(z), the term's relative error is z's own.  z = sum - 40, sums of spread 10: chains of 64 products, whose
    results are added, err by 10 u (0.09 (64 + bs / 64))^1/2 in the root mean square (u = 2^-24: an addition's rounding, of mean
    square 0.54 u^2 / 3 of a partial sum, over half the chain's length), and adding the bias by its last place's
    2^-18 / 12^1/2; the bound is a tenth more.  (One chain of 256: 1.7 times that.)"""
    g = torch.Generator().manual_seed(n + bs)
    W, u = blocks * bs, 2.0 ** -24
    r = lambda *s: torch.randn(*s, generator=g)
    proj, wi = r(1, n, 2 * W), r(blocks, bs, bs) * 10 / bs ** 0.5
    zeros, ones = torch.zeros(W), torch.ones(W, 1)
    span_start, i32 = torch.tensor([0, n], dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
    d = lambda t: t.to(DEV).contiguous()
    a, b = (torch.full((n, W), float("nan"), device=DEV) for _ in range(2))
    K().linear_recurrence_prep(d(proj), d(zeros), d(ones), d(zeros), 1, d(r(1, 8)), 8, d(torch.zeros(blocks, bs, bs)), d(wi), d(zeros),
                               d(zeros - 40), d(zeros + 0.5), i32, i32[:1], span_start, i32[:1], a, b, blocks)
    x = proj[0, :, W:].double()
    z = (x.view(n, blocks, 1, bs) @ wi.double()).reshape(n, W) - 40
    want = (1 - torch.exp(torch.tensor(-0.5, dtype=F64))).sqrt() * torch.sigmoid(z) * x
    err = (b.double().cpu() / want - 1)[(z > -64) & (z < -16) & (x != 0)]
    assert float(err.pow(2).mean().sqrt()) < 1.1 * ((10 * u) ** 2 * 0.09 * (64 + bs / 64) + 2.0 ** -36 / 12) ** 0.5


@pytest.mark.parametrize("W", [8, 72, 200])
@pytest.mark.parametrize("lens", [[1, 1, 1], [2], [63, 64, 65], [700, 1], [4, 5, 16, 1], [17, 1, 60, 1], [127, 3], [128, 1, 4, 5],
                                  [130] * 21])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("said", [False, True])
def test_recurrence_chain(W, lens, dtype, said):
    """Spans shorter than the segments are many, as long, and much longer; a state that is read and left.  Every
    split of the work: spans uncut (up to 16 tokens), 16 segments (below 128), 64, and 32 where the
    long spans are many (21 of 130 tokens at 200 channels); with and without the longest span's length."""
    g = torch.Generator().manual_seed(W)
    n, fresh = sum(lens), [i % 2 for i in range(len(lens))]
    a, b = torch.rand(n, W, generator=g) ** 0.1, torch.randn(n, W, generator=g)
    proj, y_bias, state = torch.randn(3, n, 2 * W, generator=g), torch.randn(W, generator=g), torch.randn(len(lens) + 1, 2 + W, generator=g)
    start, _, span_start, span_pos, slots = spans_of(lens, fresh)
    dev_state, out = state.to(DEV), torch.full((n, W), float("nan"), device=DEV, dtype=dtype)
    K().linear_recurrence_scan(a.to(DEV), b.to(DEV), proj.to(DEV), y_bias.to(DEV), dev_state, 2, slots, span_start,
                               span_pos, len(lens), out, longest=max(lens) if said else 0)
    y = torch.nn.functional.gelu(proj.double().sum(0)[:, :W] + y_bias.double(), approximate="tanh")
    want, state = torch.zeros(n, W, dtype=F64), state.double()
    for s in range(len(lens)):
        S = state[int(slots[s]), 2:] * (0.0 if fresh[s] else 1.0)
        for t in range(start[s], start[s + 1]):
            S = a[t].double() * S + b[t].double()
            want[t] = S * y[t]
        state[int(slots[s]), 2:] = S
    close(out, want, rel=4e-5 if dtype == torch.float32 else 5e-3)
    close(dev_state, state)


@pytest.mark.parametrize("lens", [[0, 1, 0], [0, 0, 2, 0], [3, 0], [0, 70, 0, 1], [1, 0, 40, 0, 0, 3]])
def test_recurrence_chain_with_empty_spans(lens):
    """Spans without tokens, also more spans than tokens: their states stay (or, where the span starts at
    position 0, become zero), the others' outputs and states are as without them."""
    g = torch.Generator().manual_seed(len(lens))
    n, W, fresh = sum(lens), 72, [i % 2 for i in range(len(lens))]
    a, b = torch.rand(n, W, generator=g) ** 0.1, torch.randn(n, W, generator=g)
    proj, y_bias, state = torch.randn(1, n, 2 * W, generator=g), torch.randn(W, generator=g), torch.randn(len(lens) + 1, W, generator=g)
    start, _, span_start, span_pos, slots = spans_of(lens, fresh)
    dev_state, out = state.to(DEV), torch.full((n, W), float("nan"), device=DEV)
    K().linear_recurrence_scan(a.to(DEV), b.to(DEV), proj.to(DEV), y_bias.to(DEV), dev_state, 0, slots, span_start,
                               span_pos, len(lens), out)
    y = torch.nn.functional.gelu(proj[0].double()[:, :W] + y_bias.double(), approximate="tanh")
    want, state = torch.zeros(n, W, dtype=F64), state.double()
    for s in range(len(lens)):
        S = state[int(slots[s])] * (0.0 if fresh[s] else 1.0)
        for t in range(start[s], start[s + 1]):
            S = a[t].double() * S + b[t].double()
            want[t] = S * y[t]
        state[int(slots[s])] = S
    close(out, want)
    close(dev_state, state)


SIXTEENS = [[1], [16], [17, 1, 33], [48, 15, 0, 16], [100, 3], [1] * 70 + [64]]


def delta_inputs(dk, dv, lens, fresh, seed):
    g = torch.Generator().manual_seed(seed)
    n, H, G = sum(lens), 4, 2
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    k, q = (unit(torch.randn(n, G, dk, generator=g)) for _ in range(2))
    v, beta = torch.randn(n, H, dv, generator=g), torch.rand(n, H, generator=g)
    decay = torch.rand(n, H, generator=g) ** 0.25
    decay[-1, 0] = 0.0                                                     # forgets everything
    state = torch.randn(len(lens) + 1, 8 + H * dk * dv, generator=g)
    return H, G, k, q, v, beta, decay, state, spans_of(lens, fresh)


def run_delta(dk, dv, lens, H, G, k, q, v, beta, decay, state, spans, sixteens):
    n, (_, _, span_start, span_pos, slots) = sum(lens), spans
    f = lambda t: t.to(DEV).contiguous()
    dev_state, out = f(state), torch.full((n, H * dv), float("nan"), device=DEV)
    q, k, gb, factors = f(q).view(n, -1), f(k).view(n, -1), f(torch.stack([decay, beta], dim=1)), None
    if sixteens:
        floats = K().gated_delta_factor_floats(n, len(lens), H, G, dk)
        factors = torch.full((floats,), float("nan"), device=DEV)
        K().gated_delta_factors(q, k, gb, span_start, len(lens), factors, H, G, dk)
    K().gated_delta_scan(q, k, f(v).view(n, -1), gb, out, dev_state, 8, slots, span_start, span_pos, len(lens), H, G, dk, dv,
                         factors=factors)
    return out.cpu().view(n, H, dv), dev_state.cpu()


@pytest.mark.parametrize("dk,dv", [(8, 24), (64, 16), (65, 17), (128, 40), (136, 16), (200, 8), (256, 33)])
@pytest.mark.parametrize("lens", SIXTEENS, ids=len)
def test_delta_scan_by_sixteens(dk, dv, lens):
    """Spans that end inside a sixteen, at its end and behind it, single tokens among them, more spans than a wave's lanes;
    4e-5 of the largest number is what sums of 256 + 16 rounded products of a sum near one may be off by."""
    fresh = [i % 2 for i in range(len(lens))]
    H, G, k, q, v, beta, decay, state, spans = delta_inputs(dk, dv, lens, fresh, dk + dv)
    out, after = run_delta(dk, dv, lens, H, G, k, q, v, beta, decay, state, spans, True)
    start, slots = spans[0], spans[4]
    want, want_state = torch.zeros(sum(lens), H, dv, dtype=F64), state.double()
    for s in range(len(lens)):
        slot = int(slots[s])
        S = want_state[slot, 8:].view(H, dk, dv).clone() * (0.0 if fresh[s] else 1.0)
        for t in range(start[s], start[s + 1]):
            kk, qq = (x[t].double().repeat_interleave(H // G, 0) for x in (k, q))
            S = S * decay[t].double()[:, None, None]
            u = beta[t].double()[:, None] * (v[t].double() - (S * kk[:, :, None]).sum(1))
            S = S + kk[:, :, None] * u[:, None, :]
            want[t] = (S * qq[:, :, None]).sum(1)
        want_state[slot, 8:] = S.reshape(-1)
    close(out.to(DEV), want)
    close(after.to(DEV), want_state)


@pytest.mark.parametrize("what", ["v", "k", "q", "beta", "decay", "state"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_delta_scan_by_sixteens_of_numbers_that_are_not_finite(what, value):
    """They reach what they reach when tokens are taken one by one: nothing before them, no other head of values, and behind a
    span's end no state that was finite."""
    dk, dv, lens = 72, 20, [37, 20]
    H, G, k, q, v, beta, decay, state, spans = delta_inputs(dk, dv, lens, [0, 0], 5)
    if what == "state":
        state[int(spans[4][1]), 8 + dk * dv + 3] = value                   # (second span, head 1, row 0, column 3)
    else:
        x = {"v": v, "k": k, "q": q, "beta": beta, "decay": decay}[what]
        x[21, 1] = value if x.ndim == 2 else x[21, 1]
        if x.ndim == 3:
            x[21, 1, 2] = value
    one, one_state = run_delta(dk, dv, lens, H, G, k, q, v, beta, decay, state, spans, False)
    out, after = run_delta(dk, dv, lens, H, G, k, q, v, beta, decay, state, spans, True)
    assert torch.equal(out.isfinite(), one.isfinite()) and torch.equal(after.isfinite(), one_state.isfinite())
    close(out.nan_to_num(0, 0, 0).to(DEV), one.nan_to_num(0, 0, 0).double())
    close(after.nan_to_num(0, 0, 0).to(DEV), one_state.nan_to_num(0, 0, 0).double())


@pytest.mark.parametrize("taps", [1, 2, 4, 5])
@pytest.mark.parametrize("sixteens", [False, True])
def test_scans_leave_the_convolutions_inputs(taps, sixteens):
    """In a scan's launch as in the launch of their own: spans of 0 to more tokens than the state holds, from position 0 and
    behind earlier tokens; whole numbers are copied, so the states are the same."""
    dk, dv, lens, fresh = 24, 20, [1, 2, 0, 3, 4, 0, 9, 1], [0, 1, 0, 0, 1, 1, 0, 1]
    H, G, k, q, v, beta, decay, state, spans = delta_inputs(dk, dv, lens, fresh, 3)
    n, C, (_, _, span_start, span_pos, slots) = sum(lens), 2 * G * dk + H * dv, spans
    at = 8 + H * dk * dv
    state = torch.cat([state, torch.randn(len(lens) + 1, C * (taps - 1))], dim=1)
    proj = torch.randn(2, n, C + 7, device=DEV)
    f = lambda t: t.to(DEV).contiguous()
    want, got, out = f(state), f(state), torch.empty(n, H * dv, device=DEV)
    gb, factors = f(torch.stack([decay, beta], dim=1)), None
    if sixteens:
        factors = torch.empty(K().gated_delta_factor_floats(n, len(lens), H, G, dk), device=DEV)
        K().gated_delta_factors(f(q).view(n, -1), f(k).view(n, -1), gb, span_start, len(lens), factors, H, G, dk)
    K().conv_state_update(proj, 0, C, taps, want, at, slots, span_start, span_pos, len(lens))
    K().gated_delta_scan(f(q).view(n, -1), f(k).view(n, -1), f(v).view(n, -1), gb, out, got, 8, slots, span_start, span_pos,
                         len(lens), H, G, dk, dv, factors=factors, conv=(proj, C, taps, at))
    assert torch.equal(got[:, at:], want[:, at:])


@pytest.mark.parametrize("taps", [1, 2, 4, 5])
@pytest.mark.parametrize("longest", [9, 40, 200])                      # (one segment a span, sixteen and more)
def test_linear_scan_leaves_the_convolutions_inputs(taps, longest):
    W, lens, fresh = 40, [1, 2, 0, 3, 4, longest, 0, 1], [0, 1, 0, 0, 1, 0, 1, 1]
    n = sum(lens)
    _, _, span_start, span_pos, slots = spans_of(lens, fresh)
    state = torch.randn(len(lens) + 1, W * taps + 3, device=DEV)
    proj, bias, y_bias = torch.randn(2, n, 2 * W, device=DEV), torch.randn(W, device=DEV), torch.randn(W, device=DEV)
    a, b, out = torch.rand(n, W, device=DEV), torch.randn(n, W, device=DEV), torch.empty(n, W, device=DEV)
    want, got = state.clone(), state.clone()
    K().conv_state_update(proj, W, W, taps, want, W + 3, slots, span_start, span_pos, len(lens), in_bias=bias)
    K().linear_recurrence_scan(a, b, proj, y_bias, got, 3, slots, span_start, span_pos, len(lens), out, longest=longest,
                               conv=(bias, taps, W + 3))
    assert torch.equal(got[:, W + 3:], want[:, W + 3:])


@pytest.mark.parametrize("d", [200, 1024, 2048, 4096, 5000])
@pytest.mark.parametrize("slices", [(1, 1), (2, 3)])
def test_norm_of_two_sums_without_weights(d, slices):
    """The sum in the norm's launch is the sum of a launch in front of it, rounding for rounding."""
    g = torch.Generator(device=DEV).manual_seed(d)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    n, x, w = 5, r(5, d), r(d)
    a, b, both = r(slices[0], n, d), r(slices[1], n, d), torch.empty(n, d, device=DEV)
    K().scaled_sum(both, a, 0.75, b, -1.5)
    want, got = x.clone(), x.clone()
    out, out_want = torch.empty(n, d, device=DEV, dtype=torch.bfloat16), torch.empty(n, d, device=DEV, dtype=torch.bfloat16)
    K().norm_residual(want, w, both, out=out_want, eps=1e-5)
    K().norm_residual(got, w, K().NormedPair(a, 0.75, None, b, -1.5, None), out=out, eps=1e-5)
    assert torch.equal(got, want) and torch.equal(out, out_want)


@pytest.mark.parametrize("d", [8200, 16384])
def test_norm_of_two_sums_without_weights_of_wide_rows(d):
    """Rows of which two do not fit into a launch's 64 KB of LDS: the two sums are added on the way there."""
    test_norm_of_two_sums_without_weights(d, (2, 1))


@pytest.mark.parametrize("W,spans", [(70, 3), (1100, 3), (2048, 97)])
@pytest.mark.parametrize("longest", [1, 30, 150])
def test_linear_scan_leaves_the_inputs_of_more_channels_than_a_workgroup(W, spans, longest):
    """Workgroups of 64 to 1,024 threads for the convolution's inputs, the last one not whole; 97 single tokens of 2,048 channels
    (more than twelve workgroups a CU) leave them by the chain's own threads."""
    lens = [1] * (spans - 1) + [longest]
    fresh, taps, n = [i % 2 for i in range(spans)], 4, sum(lens)
    _, _, span_start, span_pos, slots = spans_of(lens, fresh)
    state = torch.randn(spans + 1, W * taps, device=DEV)
    proj, bias, y_bias = torch.randn(1, n, 2 * W, device=DEV), torch.randn(W, device=DEV), torch.randn(W, device=DEV)
    a, b, out = torch.rand(n, W, device=DEV), torch.randn(n, W, device=DEV), torch.empty(n, W, device=DEV)
    want, got, alone = state.clone(), state.clone(), torch.empty(n, W, device=DEV)
    K().conv_state_update(proj, W, W, taps, want, W, slots, span_start, span_pos, spans, in_bias=bias)
    K().linear_recurrence_scan(a, b, proj, y_bias, want, 0, slots, span_start, span_pos, spans, alone, longest=longest)
    K().linear_recurrence_scan(a, b, proj, y_bias, got, 0, slots, span_start, span_pos, spans, out, longest=longest,
                               conv=(bias, taps, W))
    assert torch.equal(got, want) and torch.equal(out, alone)


@pytest.mark.parametrize("d", [4, 7, 1020, 1026, 2048, 2046, 3000, 4093])
@pytest.mark.parametrize("slices,paired", [(1, 0), (3, 0), (2, 1), (1, 2)])
def test_norm_behind_a_sub_layer_whole_and_odd_rows(d, slices, paired):
    """Rows that are read sixteen bytes at a time and rows (by their length, or by where they start) that are not, over the edges of a
    thread's elements; slices, two sums side by side as they are (1) or normed (2), and the next norm's rows.  Sums of up to 4,093
    squares in 32 bits: 1e-6 of the result."""
    k = K()
    g = torch.Generator().manual_seed(d + slices)
    n, eps = 3, 1e-5
    odd = 1 if d in (1020, 3000) else 0            # a first element that is not on 16 bytes
    def dev(t):
        flat = torch.empty(t.numel() + odd, device="cuda")
        flat[odd:] = t.flatten().cuda()
        return flat[odd:].view(t.shape)
    x, w, w2 = torch.randn(n, d, generator=g), torch.randn(d, generator=g), torch.randn(d, generator=g)
    a, b = torch.randn(slices, n, d, generator=g), torch.randn(2, n, d, generator=g)
    wa, wb = torch.randn(d, generator=g), torch.randn(d, generator=g)
    norm = lambda v: v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps)
    A, B = a.double().sum(0), b.double().sum(0)
    delta = A if paired == 0 else 0.75 * A - 1.5 * B if paired == 1 else 0.75 * wa.double() * norm(A) - 1.5 * wb.double() * norm(B)
    want = x.double() + 0.6 * w.double() * norm(delta)
    xd, out = dev(x), torch.empty(n, d, device="cuda")
    arg = dev(a) if paired == 0 else k.NormedPair(dev(a), 0.75, dev(wa) if paired == 2 else None, dev(b), -1.5, dev(wb) if paired == 2 else None)
    k.norm_residual(xd, dev(w), arg, out=out, eps=eps, mult=0.6, next_weight=dev(w2))
    for got, ref in ((xd, want), (out, norm(want) * w2.double())):
        err = (got.double().cpu() - ref).norm() / ref.norm()
        assert err < 1e-6, float(err)


@pytest.mark.parametrize("dk,dv", [(8, 24), (64, 16), (65, 20), (128, 40), (136, 16), (200, 8), (256, 36)])
@pytest.mark.parametrize("per_channel", [False, True])
def test_delta_scan_of_single_tokens_where_rows_are_whole_pieces(dk, dv, per_channel):
    """Spans of one token whose state lies on 16 bytes: against the same states four bytes further, which go token by token.  A sum of dk
    products in another order, and what hangs on it, differs by dk 2^-23 of the magnitudes, here at most a few units."""
    g = torch.Generator().manual_seed(dk * dv)
    n, H, G = 5, 4, 2
    unit = lambda t: (t / t.norm(dim=-1, keepdim=True)).view(n, -1).to(DEV).contiguous()
    k, q = (unit(torch.randn(n, G, dk, generator=g)) for _ in range(2))
    v, dec = torch.randn(n, H * dv, generator=g).to(DEV), torch.rand(n, H * dk, generator=g).to(DEV)
    gb = torch.rand(n, 2, H, generator=g).to(DEV)
    fill = torch.randn(n + 1, H * dk * dv, generator=g).to(DEV)
    _, _, span_start, span_pos, slots = spans_of([1] * n, [0, 1, 0, 0, 1])
    got = {}
    for at in (4, 5):
        state = torch.zeros(n + 1, 8 + H * dk * dv, device=DEV)
        state[:, at:at + H * dk * dv] = fill
        out = torch.full((n, H * dv), float("nan"), device=DEV)
        K().gated_delta_scan(q, k, v, gb, out, state, at, slots, span_start, span_pos, n, H, G, dk, dv, dec if per_channel else None)
        assert not state[:, :at].any() and not state[:, at + H * dk * dv:].any()
        got[at] = out, state[:, at:at + H * dk * dv]
    for one, other in zip(got[4], got[5]):
        assert (one - other).abs().max() <= dk * 2.0 ** -23 * 8


@pytest.mark.parametrize("dk,dv", [(64, 128), (128, 130), (200, 40), (256, 300)])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("nsplit", [1, 3])
def test_delta_preparation(dk, dv, taps, nsplit):
    """Convolution, SiLU and unit norms against 64 bits: spans that begin inside a token's window, behind earlier tokens and at position 0;
    heads of one, of two and of more than two channels a lane."""
    g = torch.Generator().manual_seed(dk + taps)
    lens, fresh, H, G = [1, 1, 2, 5, 1], [0, 1, 0, 1, 0], 2, 1
    n, QK, HV = sum(lens), G * dk, H * dv
    C = 2 * QK + HV
    start, token, span_start, span_pos, slots = spans_of(lens, fresh)
    proj = torch.randn(nsplit, n, C + 2 * H + HV + 3, generator=g)
    w, a_log, dt = torch.randn(C, taps, generator=g), torch.randn(H, generator=g), torch.randn(H, generator=g)
    state = torch.randn(len(lens) + 1, 3 + C * (taps - 1), generator=g)
    f = lambda t: t.to(DEV).contiguous()
    qn, kn, vv, gate = (torch.full((n, m), float("nan"), device=DEV) for m in (QK, QK, HV, HV))
    gb = torch.full((n, 2, H), float("nan"), device=DEV)
    K().gated_delta_prep(f(proj), f(w), taps, f(state), 3, f(a_log), f(dt), token, slots, span_start, span_pos, qn, kn, vv, gb, gate, H, G, dk, dv)
    x = proj.double().sum(0)
    y = torch.zeros(n, C, dtype=F64)
    for s in range(len(lens)):
        before = state[int(slots[s]), 3:].double().view(C, taps - 1).T * (0.0 if fresh[s] else 1.0)
        rows = torch.cat([before, x[start[s]:start[s + 1], :C]])
        for t in range(lens[s]):
            y[start[s] + t] = (rows[t:t + taps] * w.double().T).sum(0)
    y = torch.nn.functional.silu(y)
    unit = lambda t: t / (t.view(n, G, dk).norm(dim=-1, keepdim=True).square() + 1e-6).sqrt().expand(n, G, dk).reshape(n, QK)
    close(qn, unit(y[:, :QK]) * dk ** -0.5)
    close(kn, unit(y[:, QK:2 * QK]))
    close(vv, y[:, 2 * QK:])
    close(gate, torch.nn.functional.silu(x[:, C + 2 * H:C + 2 * H + HV]))
    close(gb[:, 1], torch.sigmoid(x[:, C:C + H]))
    close(gb[:, 0], torch.exp(-a_log.double().exp() * torch.nn.functional.softplus(x[:, C + H:C + 2 * H] + dt.double())))
