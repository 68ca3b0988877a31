"""rrl_policy_prepare, rrl_targets_status and rrl_policy_forward / _backward
through the C ABI (MI355X): the stored status word, and the split of long
sequences, against plain torch in float64.

Bars: float32 sums of n terms in another order, 1e-6 relative on means and
1e-5 on gradients.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from rosellm_amd import _native as nat
from rosellm_amd import roserlhf as R
from rosellm_amd.roserlhf import losses as L
from rosellm_amd.rosetrainer import cross_entropy

pytestmark = pytest.mark.gpu


def _view(t):
    return nat.rows_view(t, *t.shape)[0]


def _targets_status(t, V, params=None, word=None):
    word = torch.full((1,), 77, dtype=torch.int32, device=t.device) if word is None else word
    part = torch.empty(nat.lib().rrl_targets_workspace_bytes(), dtype=torch.uint8, device=t.device)
    nat.call("rrl_targets_status", ctypes.byref(params or nat.RrlPolicyParams()), *t.shape, V,
             _view(t), part.data_ptr(), word.data_ptr(), nat.stream_ptr(t.device))
    torch.cuda.synchronize()
    return int(word.item())


@pytest.mark.parametrize("n", [1, 1023, 1025, 16384, 16385, 70000])
@pytest.mark.parametrize("bad", [None, 0, -1])
def test_targets_status(device, n, bad):
    """One workgroup up to 16384 tokens, parts and a combine beyond; the word
    is overwritten whatever it held."""

    t = torch.randint(0, 50, (1, n), device=device)
    if bad is not None:
        t[0, bad] = 50 if bad == 0 else -1
    want = 0 if bad is None else nat.FLAG_TARGET_RANGE
    assert _targets_status(t, 50) == want
    host = torch.full((1,), 77, dtype=torch.int32, pin_memory=True)
    assert _targets_status(t, 50, word=host) == want
    nll = nat.RrlPolicyParams(kind=nat.OBJ_NLL, ignore_index=-1)
    assert _targets_status(t, 50, nll) == (want if bad == 0 else 0)


@pytest.mark.parametrize("B,T", [(1, 1), (3, 255), (2, 257), (5, 2048), (300, 9), (2, 8192)])
@pytest.mark.parametrize("kind", [nat.OBJ_PPO, nat.OBJ_SAPO, nat.OBJ_GSPO])
def test_prepare_and_forward(device, B, T, kind):
    """Row coefficients, records and scalars where a sequence takes one part,
    all eight, and a remainder; more and fewer sequences than 256."""

    g = torch.Generator(device=device).manual_seed(B * T + kind)
    t = torch.randint(0, 100, (B, T), device=device, generator=g)
    old = -3.0 + torch.randn(B, T, device=device, generator=g)
    cur = old + 0.1 * torch.randn(B, T, device=device, generator=g)
    adv = 0.5 + torch.randn(B, T, device=device, generator=g)
    mask = torch.rand(B, T, device=device, generator=g) < 0.7
    mask[:, 0] = True
    p = L._params(kind, clip_low=0.2, clip_high=0.3, mask_is_weight=kind == nat.OBJ_PPO)
    gspo = kind == nat.OBJ_GSPO
    ws = torch.empty(nat.lib().rrl_policy_workspace_bytes(B, nat.F32), dtype=torch.uint8,
                     device=device)
    rec = torch.empty(nat.lib().rrl_fused_records_bytes(B, T), dtype=torch.uint8, device=device)
    coef = torch.empty(B, device=device)
    word = torch.full((1,), 77, dtype=torch.int32, device=device)

    def prepare(tt, mm):
        nat.call("rrl_policy_prepare", ctypes.byref(p), B, T, 100, _view(tt), _view(old),
                 _view(adv), _view(mm), nat.F32, None if gspo else coef.data_ptr(),
                 None if gspo else rec.data_ptr(), ws.data_ptr(), word.data_ptr(),
                 nat.stream_ptr(device))
        return int(word.item())

    bad = t.clone()
    bad[-1, -1] = 100
    assert prepare(bad, mask) == nat.FLAG_TARGET_RANGE
    none = mask.clone()
    none[-1] = False
    want = nat.FLAG_EMPTY_ROW if kind != nat.OBJ_PPO else (nat.FLAG_EMPTY_MASK if B == 1 else 0)
    assert prepare(t, none) == want
    assert prepare(t, mask) == 0
    m = mask.double()
    if not gspo:
        r = rec[:16 * B * T].view(torch.float32).view(B, T, 4)
        assert torch.equal(r[..., 0].contiguous().view(torch.int32), t.int())
        assert torch.equal(r[..., 1], old) and torch.equal(r[..., 2], adv)
        assert torch.equal(r[..., 3], mask.float())
        wc = 1.0 / (m.sum(1) * B) if kind == nat.OBJ_SAPO else (1.0 / m.sum()).expand(B)
        assert torch.allclose(coef.double(), wc, rtol=1e-6)
    if kind != nat.OBJ_PPO:
        return
    outs = [torch.empty((), device=device) for _ in range(4)] + [
        torch.empty((), dtype=torch.float64, device=device)]
    nat.call("rrl_policy_forward", ctypes.byref(p), B, T, _view(cur), _view(old), _view(adv),
             _view(mask), nat.F32, ws.data_ptr(), ctypes.byref(nat.scalars(outs)), None, None,
             word.data_ptr(), nat.stream_ptr(device))
    assert int(word.item()) == 0
    lp = cur.double().requires_grad_()
    rho = (lp - old.double()).exp()
    obj = (torch.minimum(rho * adv, rho.clamp(0.8, 1.3) * adv) * m).sum() / m.sum()
    mean = (rho * m).sum() / m.sum()
    scale = ((rho * adv).abs() * m).sum().item() / m.sum().item()
    assert abs(outs[0].item() - obj.item()) <= 1e-6 * scale
    assert abs(outs[3].item() - mean.item()) <= 1e-6 * mean.item()
    assert outs[4].item() == -outs[0].item()
    # upstream gradients of the loss, the objective and the mean ratio at once
    g4 = [torch.tensor(0.5, device=device), None, None, torch.tensor(0.25, device=device),
          torch.tensor(2.0, dtype=torch.float64, device=device)]
    grad = torch.empty(B, T, device=device)
    nat.call("rrl_policy_backward", ctypes.byref(p), B, T, _view(cur), _view(old), _view(adv),
             _view(mask), nat.F32, ws.data_ptr(), ctypes.byref(nat.scalars(g4)), None,
             grad.data_ptr(), nat.stream_ptr(device))
    (want,) = torch.autograd.grad((0.5 - 2.0) * obj + 0.25 * mean, lp)
    assert torch.allclose(grad.double(), want, rtol=1e-5, atol=1e-6 * want.abs().max().item())


@pytest.mark.parametrize("objective", ["gspo", "gspo_token"])
def test_sequences_without_positions(device, objective):
    """[B, 0]: no sequence has an action token, fused as composed."""

    B, V = 3, 16
    x = torch.zeros(B, 0, V, device=device)
    t = torch.zeros(B, 0, dtype=torch.int64, device=device)
    z = torch.zeros(B, 0, device=device)
    adv = torch.zeros(B, device=device) if objective == "gspo" else z
    mask = torch.zeros(B, 0, dtype=torch.bool, device=device)
    composed = R.gspo_policy_loss if objective == "gspo" else R.gspo_token_policy_loss
    with pytest.raises(ValueError, match="at least one action token"):
        composed(R.gather_token_logprobs(x, t), z, adv, mask, clip_low=0.1, clip_high=0.1)
    with pytest.raises(ValueError, match="at least one action token"):
        R.fused_policy_loss(x, t, z, adv, mask, objective=objective, clip_low=0.1)


def test_token_objectives_without_positions(device):
    """[B, 0] through the single-pass objectives: the composed loss's error,
    and torch's own values for a cross-entropy over nothing."""

    x = torch.zeros(3, 0, 16, device=device)
    t = torch.zeros(3, 0, dtype=torch.int64, device=device)
    z = torch.zeros(3, 0, device=device)
    with pytest.raises(ValueError, match="empty mask"):
        R.fused_policy_loss(x, t, z, z, t.bool(), clip_low=0.1)
    with pytest.raises(ValueError, match="at least one action token"):
        R.fused_policy_loss(x, t, z, z, t.bool(), objective="sapo", tau_positive=1.0,
                            tau_negative=1.0)
    assert torch.isnan(cross_entropy(x, t))
    assert cross_entropy(x, t, reduction="sum").item() == 0.0


def _flagging_calls(device, B=64, T=2048):
    """(entry point's call on a status address, its bit) for the entry points
    that OR a bit: every token, row or mask of the inputs is a bad one."""

    x = torch.ones(B, T, device=device)
    none = torch.zeros(B, T, dtype=torch.bool, device=device)
    live = ~none
    ids = torch.full((B, T), 7, dtype=torch.int64, device=device)
    ws = torch.empty(nat.lib().rrl_reduce_workspace_bytes(B * T), dtype=torch.uint8, device=device)
    out, cnt = torch.empty_like(x), torch.empty_like(x)
    s = lambda: nat.stream_ptr(device)  # noqa: E731
    v = _view
    return [
        (lambda p: nat.call("rrl_masked_whiten", B, T, v(x), v(none), 1e-8, 1, nat.F32,
                            ws.data_ptr(), out.data_ptr(), nat.F32, p, s()), nat.FLAG_EMPTY_MASK),
        (lambda p: nat.call("rrl_masked_mean_fwd", B, T, v(x), v(none), nat.F32, ws.data_ptr(),
                            out.data_ptr(), p, s()), nat.FLAG_EMPTY_MASK),
        (lambda p: nat.call("rrl_sequence_log_ratio_fwd", B, T, v(x), v(x), v(none), 1, nat.F32,
                            out.data_ptr(), cnt.data_ptr(), p, s()), nat.FLAG_EMPTY_ROW),
        (lambda p: nat.call("rrl_broadcast_turn", B, 1, T, nat.rows_view(x[:, :1], B, 1)[0], v(ids),
                            v(live), cnt.data_ptr(), nat.F32, p, s()), nat.FLAG_INVALID_TURN),
    ]


def test_status_word_shared_between_streams(device):
    """A device status word takes bits from calls on several streams at once and
    keeps those already set; a host word (RRL_STATUS_HOST) is set without
    atomics; a null one is not written."""

    calls = _flagging_calls(device)
    for f, bit in calls:
        word = torch.full((1,), 64, dtype=torch.int32, device=device)
        f(word.data_ptr())
        f(None)
        assert int(word.item()) == 64 | bit
        with nat.HostStatus(zero=True) as host:
            f(host.ptr)
            host.record(device)
            assert host.read() == bit
    # different bits from the last two and the first, each on its own stream
    (a, ab), (b, bb), (c, cb) = calls[0], calls[2], calls[3]
    streams = [torch.cuda.Stream(device) for _ in range(3)]
    words = torch.zeros(50, dtype=torch.int32, device=device)
    torch.cuda.synchronize()
    for i in range(words.numel()):
        for f, st in zip((a, b, c), streams):
            with torch.cuda.stream(st):
                f(words[i:].data_ptr())
    torch.cuda.synchronize()
    assert words.tolist() == [ab | bb | cb] * words.numel()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_inplace_errors_leave_the_logits(device, dtype):
    """A bad target id or an empty mask raises before the logits are
    overwritten."""

    B, T, V = 2, 5, 4096
    x = torch.randn(B, T, V, device=device).to(dtype)
    keep = x.clone()
    t = torch.randint(0, V, (B, T), device=device)
    old = adv = torch.zeros(B, T, device=device)
    mask = torch.ones(B, T, dtype=torch.bool, device=device)
    bad = t.clone()
    bad[-1, -1] = V
    kw = dict(clip_low=0.2, inplace=True)
    with pytest.raises(RuntimeError, match="index out of bounds"):
        R.fused_policy_loss(x, bad, old, adv, mask, **kw)
    assert torch.equal(x, keep)
    with pytest.raises(ValueError, match="empty mask"):
        R.fused_policy_loss(x, t, old, adv, torch.zeros_like(mask), **kw)
    assert torch.equal(x, keep)
    with pytest.raises(IndexError):
        cross_entropy(x, bad, inplace=True)
    assert torch.equal(x, keep)
