"""The row kernels' variants at the edges of their ranges (MI355X).

A row's length and the number of rows choose how many lanes hold a row and how
many 16-byte slabs each lane carries.  Each case sits on, or one vector past,
the last length of a variant, with few and with many rows, through
``fused_policy_loss`` (mode 2) and ``gather_token_logprobs`` with its backward,
against plain torch in float64.

Bars: float32 log-probs and gradients 1e-5 relative (1e-5 of |g| per row);
bfloat16 gradients 2^-8 + 1e-5 per row in the 2-norm: rounding to 8 significant
bits moves an element by at most 2^-8 of itself, and a row may be one element.
"""

from __future__ import annotations

import pytest
import torch

from rosellm_amd import roserlhf as R

pytestmark = pytest.mark.gpu


def _rows(seed, T, V, dtype, device):
    g = torch.Generator(device=device).manual_seed(seed)
    x = (torch.randn(1, T, V, device=device, generator=g) * 3.0).to(dtype)
    t = torch.randint(0, V, (1, T), device=device, generator=g)
    # targets on the row's first and last elements too
    t[0, 0], t[0, -1] = 0, V - 1
    up = torch.randn(1, T, device=device, generator=g)
    return x, t, up


def _want(x, t, up):
    """float64 log-probs and d logits for d loss / d logp = up."""

    xd = x.double()
    lse = torch.logsumexp(xd, dim=-1, keepdim=True)
    lp = xd.gather(-1, t[..., None]) - lse
    dl = -up.double()[..., None] * torch.exp(xd - lse)
    dl.scatter_(-1, t[..., None], -up.double()[..., None] * torch.expm1(lp))
    return lp[..., 0], dl


def _row_err(got, want):
    d = (got.double() - want).norm(dim=-1)
    return (d / want.norm(dim=-1).clamp_min(1e-30)).max().item()


def _check(x, t, up, got_lp, got_dl):
    lp, dl = _want(x, t, up)
    assert torch.allclose(got_lp.double(), lp, rtol=1e-5, atol=1e-6)
    # every row's gradient carries |up| at its target at least once
    if x.dtype == torch.float16:
        # 11 significant bits, and below 2^-14 half a subnormal step (2^-25)
        # per element whatever its size
        d = (got_dl.double() - dl).abs()
        assert bool((d <= dl.abs() * (2.0 ** -11 + 1e-5) + 2.0 ** -25).all())
        return
    bar = 2.0 ** -8 + 1e-5 if x.dtype == torch.bfloat16 else 1e-5
    assert _row_err(got_dl, dl) <= bar


def _run(x, t, up):
    """The composed pass and the fused pass (old log-probs = the row's own, so
    every ratio is 1 and d loss / d logp = -adv / n exactly inside the clip)."""

    T = x.shape[1]
    xg = x.clone().requires_grad_()
    lp = R.gather_token_logprobs(xg, t)
    (dl,) = torch.autograd.grad(lp, xg, grad_outputs=up)
    _check(x, t, up, lp.detach(), dl)
    mask = torch.ones_like(t, dtype=torch.bool)
    out, lp2 = R.fused_policy_loss(xg, t, lp.detach(), up, mask, clip_low=0.2,
                                   return_logprobs=True)
    (dl2,) = torch.autograd.grad(out.loss, xg)
    _check(x, t, -up / T, lp2, dl2)


# vectors per row: the last length of each variant and one past it
EDGES = [128, 129, 256, 257, 384, 512, 513, 640, 641, 1024, 1025, 1280, 1536, 1537, 1792, 2048,
         2049, 2560, 3072, 3073, 3584, 3585]


@pytest.mark.parametrize("nvec", EDGES)
@pytest.mark.parametrize("rows", [37, 2047, 2048, 2300])
def test_short_rows(device, nvec, rows):
    """Whole 128-byte rows (nvec a multiple of 8) and rows whose body starts
    off a 128-byte boundary."""

    V = 8 * nvec
    print(f"[row-variants] bf16 V={V} rows={rows}", flush=True)
    _run(*_rows(nvec + rows, rows, V, torch.bfloat16, device))


LONG_BF16 = [4096, 4104, 5120, 6144, 6656, 6664, 7168, 8192, 8200, 9216, 9224, 12288, 13312, 14336,
             14344, 16384, 18432, 18440, 19456, 19464, 20480]
LONG_F32 = [512, 520, 6656, 7168, 7176, 8192, 8200]


@pytest.mark.parametrize("dtype,nvec", [(torch.bfloat16, n) for n in LONG_BF16]
                         + [(torch.float32, n) for n in LONG_F32])
@pytest.mark.parametrize("rows", [5, 530])
def test_long_rows(device, dtype, nvec, rows):
    V = nvec * (8 if dtype == torch.bfloat16 else 4)
    print(f"[row-variants] {dtype} V={V} rows={rows}", flush=True)
    _run(*_rows(nvec + rows, rows, V, dtype, device))


@pytest.mark.parametrize("nvec", [512, 1024, 3072, 4096, 16032, 18992])
def test_float16_every_element(device, nvec):
    """Every element of float16 rows (their kernels write a store's registers
    soonest after it)."""

    print(f"[row-variants] f16 V={8 * nvec}", flush=True)
    _run(*_rows(nvec, 2100 if nvec < 8000 else 530, 8 * nvec, torch.float16, device))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [1, 7, 2001, 4099, 8197, 16387, 24581])
def test_odd_rows(device, dtype, V):
    """Head and tail elements beside the slabs, at 2300 rows."""

    print(f"[row-variants] {dtype} odd V={V}", flush=True)
    _run(*_rows(V, 2300, V, dtype, device))


@pytest.mark.parametrize("dtype,V", [(torch.float32, v) for v in (81924, 81925, 151936, 163853)]
                         + [(torch.bfloat16, v) for v in (163848, 163853, 256000)])
@pytest.mark.parametrize("rows", [3, 300])
def test_rows_past_the_registers(device, dtype, V, rows):
    print(f"[row-variants] {dtype} V={V} rows={rows}", flush=True)
    _run(*_rows(V + rows, rows, V, dtype, device))


@pytest.mark.parametrize("nvec", [511, 512, 513, 768, 769, 3072, 3073])
@pytest.mark.parametrize("rows", [255, 256])
def test_forward_lengths(device, nvec, rows):
    """The streaming forward's lane counts and depth remainders (four slabs of
    128 to 1024 lanes), log-probs of a masked-out row 0."""

    V = 8 * nvec + (nvec % 3)
    print(f"[row-variants] forward V={V} rows={rows}", flush=True)
    x, t, _ = _rows(nvec, rows, V, torch.float16, device)
    x[0, 1, V // 2] = -float("inf")
    lp, _ = _want(x, t, torch.ones_like(t, dtype=torch.float32))
    got = R.gather_token_logprobs(x, t)
    assert torch.allclose(got.double(), lp, rtol=1e-5, atol=1e-6)
    live = torch.rand(1, rows, device=device) < 0.5
    old, adv = lp.float() + 0.01, torch.ones_like(got)
    live[0, :2] = True
    a = R.fused_policy_loss(x, t, old, adv[:, 0], live, objective="gspo", clip_low=0.2)
    b = R.fused_policy_loss(x, t, old, adv[:, 0], live, objective="gspo", clip_low=0.2,
                            skip_masked_rows=True)
    assert torch.equal(a.loss, b.loss)
