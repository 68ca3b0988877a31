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
