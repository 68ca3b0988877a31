"""Logits near the ends of the 16-bit formats' range through the register-resident
sweep (MI355X), against plain torch in float64.

A row's log-sum-exp may be far larger than its digits after the point: at 1e8
float32 steps by 8, at 3e38 by 2e31.  The gradient g * (onehot - softmax) needs
the distances from the row's maximum, which are exact, and not the sum itself.

Bars: bfloat16 rounds an element by at most 2^-8 of itself, float16 by 2^-11
(half a subnormal step, 2^-25, below 2^-14); float32 arithmetic adds 1e-5.
"""

from __future__ import annotations

import pytest
import torch

from rosellm_amd import roserlhf as R
from rosellm_amd.rosetrainer import cross_entropy

pytestmark = pytest.mark.gpu

# on both sides of 128, where the sweep changes how it forms the exponent, and up
# to the formats' last values
TOPS = [(torch.bfloat16, v) for v in (100.0, 200.0, 1.0e8, 1.0e20, 2.2e38, 3.0e38)]
TOPS += [(torch.float16, v) for v in (100.0, 200.0, 6.0e4)]
VOCABS = [4096, 4099, 151936]  # whole vectors, head and tail elements, 19 slabs


def _rows(dtype, V, device):
    g = torch.Generator(device=device).manual_seed(V)
    x = 3.0 * torch.randn(1, 6, V, device=device, generator=g)
    t = torch.randint(0, V, (1, 6), device=device, generator=g)
    return x.to(dtype), t


def _near(got, want, dtype):
    rel, tiny = (2.0 ** -8, 0.0) if dtype == torch.bfloat16 else (2.0 ** -11, 2.0 ** -25)
    err = (got.double() - want).abs()
    assert torch.isfinite(got).all()
    assert bool((err <= want.abs() * (rel + 1e-5) + tiny + 1e-30).all()), err.max().item()


@pytest.mark.parametrize("dtype,top", TOPS)
@pytest.mark.parametrize("V", VOCABS)
def test_maximum_off_the_label(device, dtype, top, V):
    """d loss / d logits is 1/n at the row's maximum, whatever its size."""

    print(f"[value-range] {dtype} top={top} V={V}", flush=True)
    x, t = _rows(dtype, V, device)
    x[0, 2, V // 3], t[0, 2] = top, V - 1
    x[0, 4, 0], t[0, 4] = -top, 0  # a label far below the row
    x[0, 5, V - 2:] = top  # two maxima, one the label
    t[0, 5] = V - 1
    want = torch.softmax(x.double(), dim=-1)
    want.scatter_add_(-1, t[..., None], -torch.ones_like(want[..., :1]))
    xg = x.clone().requires_grad_()
    (dl,) = torch.autograd.grad(cross_entropy(xg, t, reduction="sum"), xg)
    _near(dl, want, dtype)
    buf = x.clone()
    loss = cross_entropy(buf.requires_grad_(), t, reduction="sum", inplace=True)
    assert torch.equal(buf.detach(), dl) and not torch.isnan(loss)


@pytest.mark.parametrize("dtype,top", TOPS)
@pytest.mark.parametrize("V", VOCABS)
@pytest.mark.parametrize("objective", ["clipped", "sapo"])
def test_tied_maxima(device, dtype, top, V, objective):
    """Two entries tie at the maximum and one is the target: log-prob -log 2,
    half the gradient on each."""

    print(f"[value-range] {objective} {dtype} top={top} V={V}", flush=True)
    x, t = _rows(dtype, V, device)
    x[0, 1, V // 2] = x[0, 1, V - 1] = top
    t[0, 1] = V - 1
    lp = torch.log_softmax(x.double(), dim=-1)
    old = lp.gather(-1, t[..., None])[..., 0].float()
    adv = torch.tensor([[0.5, -1.25, 2.0, 0.75, -0.3, 1.0]], device=device)
    mask = torch.ones_like(t, dtype=torch.bool)
    kw = dict(clip_low=0.2) if objective == "clipped" else dict(tau_positive=1.0,
                                                                tau_negative=1.0)
    xg = x.clone().requires_grad_()
    out, got = R.fused_policy_loss(xg, t, old, adv, mask, objective=objective,
                                   return_logprobs=True, **kw)
    (dl,) = torch.autograd.grad(out.loss, xg)
    assert torch.allclose(got, old, rtol=1e-5, atol=1e-6)
    # ratio 1: d loss / d logp = -adv / n for the clipped loss and for SAPO's
    # gate at its centre
    g = -adv.double()[..., None] / 6
    want = -g * lp.exp()
    want.scatter_add_(-1, t[..., None], g)
    _near(dl, want, dtype)
    buf = x.clone()
    out_i = R.fused_policy_loss(buf.requires_grad_(), t, old, adv, mask, objective=objective,
                                inplace=True, **kw)
    assert torch.equal(buf.detach(), dl) and torch.equal(out_i.loss, out.loss)


@pytest.mark.parametrize("top", [1.0e8, 3.0e38])
def test_lm_head_logits(device, top):
    """The chunked LM head over logits as large, one tied with the target's:
    d weight = d logits^T @ hidden."""

    V, H = 512, 64
    g = torch.Generator(device=device).manual_seed(5)
    h = torch.zeros(1, 4, H, device=device)
    h[0, :, 0] = torch.tensor([1.0, 1.0, 0.0, 0.0], device=device)
    h[0, :, 1:] = 0.01 * torch.randn(4, H - 1, device=device, generator=g)
    w = torch.zeros(V, H, device=device)
    w[3, 0] = w[7, 0] = top
    h, w = h.bfloat16().requires_grad_(), w.bfloat16().requires_grad_()
    t = torch.tensor([[3, 9, 3, 9]], device=device)
    x = (h.detach().double()[0] @ w.detach().double().t()).bfloat16().double()
    lp = torch.log_softmax(x, dim=-1)
    old = lp.gather(-1, t[0][:, None]).float().view(1, 4).clamp_min(-80.0)
    adv = torch.tensor([[1.0, 0.0, -0.5, 2.0]], device=device)
    mask = torch.ones_like(t, dtype=torch.bool)
    out = R.fused_linear_policy_loss(h, w, t, old, adv, mask, objective="clipped", clip_low=0.2)
    dh, dw = torch.autograd.grad(out.loss, (h, w))
    assert torch.isfinite(dw).all()
    up = -adv.double()[0][:, None] / 4
    dl = -up * lp.exp()
    dl.scatter_add_(-1, t[0][:, None], up)
    want = dl.t() @ h.detach().double()[0]
    # d logits and the product are each rounded to bfloat16
    assert ((dw.double() - want).abs() <= 2.0 ** -6 * want.abs().max()).all()


def test_rerun_flag_launches_nothing(device):
    """RRL_POLICY_RERUN_FAST_RANGE (C callers): the first call's outputs stand
    and its status word stays clear; without one the call is refused."""

    import ctypes

    from rosellm_amd import _native as nat
    from rosellm_amd.roserlhf import losses as L

    B, T, V = 1, 6, 4096
    x, t = _rows(torch.bfloat16, V, device)
    x[0, 2, 9] = 3.0e38
    t[0, 2] = 11
    z, one = torch.zeros(B, T, device=device), torch.ones(B, T, device=device)
    mask = torch.ones_like(t, dtype=torch.bool)
    coef = torch.full((B,), 1.0 / T, device=device)
    rec = torch.empty(nat.lib().rrl_fused_records_bytes(B, T), dtype=torch.uint8, device=device)
    lp, lse, dl = torch.empty_like(z), torch.empty_like(z), torch.empty_like(x)
    status = nat.new_status(device)
    p = L._params(nat.OBJ_PPO, clip_low=0.2, clip_high=0.2, mask_is_weight=True)

    def call(flags, word):
        p.flags = flags
        v = [nat.rows_view(q, B, T)[0] for q in (t, z, one, mask)]
        nat.call("rrl_fused_logprob_policy", ctypes.byref(p), x.data_ptr(), nat.BF16, B, T, V,
                 T * V, V, *v, coef.data_ptr(), rec.data_ptr(), lp.data_ptr(), lse.data_ptr(),
                 dl.data_ptr(), nat.BF16, T * V, V, word, nat.stream_ptr(device))

    call(0, status.data_ptr())
    first = (lp.clone(), lse.clone(), dl.clone())
    assert int(status.item()) == 0 and torch.isfinite(dl).all()
    call(nat.POLICY_RERUN_FAST_RANGE, status.data_ptr())
    assert all(torch.equal(a, b) for a, b in zip(first, (lp, lse, dl)))
    assert int(status.item()) == 0
    with pytest.raises(RuntimeError, match="status word"):
        call(nat.POLICY_RERUN_FAST_RANGE, None)
