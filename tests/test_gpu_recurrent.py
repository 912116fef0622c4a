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
