"""The calls whose speed counts: training steps, scoring passes, estimators and
rollout sampling, each through the package's public entry points.

``listed()`` holds one case per path at a size taken from this repository's
configurations and tests (or a generic one); ``draw()`` gives further cases of
the same ranges.  ``prepare`` makes what a program has in hand before the
call, ``run`` is one pass, ``work`` the bytes and operations the pass cannot
do without, ``tolerance`` how far two correct implementations at the same
precision may lie apart and ``exact`` the outputs in 64 bits from plain torch.
"""

import math

import torch

from rosellm_amd import roserlhf as R
from rosellm_amd.roseinfer import sample_next_token_batch
from rosellm_amd.rosetrainer import causal_lm_loss

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZES = {"bf16": 2, "f16": 2, "f32": 4}
GROUP = 4  # rollouts per prompt

# Sampler settings: (temperature, top_k, top_p, do_sample, log q asked for).
SETTINGS = {
    "default": (1.0, 0, 1.0, True, True),
    "default_no_q": (1.0, 0, 1.0, True, False),
    "topk_topp": (0.7, 50, 0.9, True, True),
    "topp": (1.0, 0, 0.9, True, True),
    "greedy": (1.0, 0, 1.0, False, True),
}

# Objective keyword arguments of bench.py's configurations.
OBJECTIVES = {
    "clipped": dict(clip_low=0.2, clip_high=0.28),
    "sao": dict(clip_low=0.2, clip_high=0.28),
    "sapo": dict(tau_positive=1.0, tau_negative=1.05),
    "gspo": dict(clip_low=3e-4, clip_high=4e-4),
}


def listed():
    return [
        # The drop-in composition on a toy policy: gather_token_logprobs, the
        # group statistics, the clipped loss and autograd.  Launches and the
        # host count here, not bytes.
        dict(name="toy_composed_f32", kind="composed", B=16, T=32, V=4096, dtype="f32",
             objective="clipped"),
        # The GRPO toy configuration: 32 x 128 tokens of a 50257-entry
        # vocabulary in float32 (rows off every 16-byte boundary).
        dict(name="grpo_f32_50257", kind="fused", B=32, T=128, V=50257, dtype="f32",
             objective="clipped", skip=False),
        # One micro-batch of the headline GRPO step: 16 x 1024 tokens of
        # 151936 bfloat16 logits.  The largest case by bytes.
        dict(name="grpo_bf16_151936", kind="fused", B=16, T=1024, V=151936, dtype="bf16",
             objective="clipped", skip=False),
        # A small-vocabulary policy in mixed precision.
        dict(name="sao_bf16_32000", kind="fused", B=16, T=512, V=32000, dtype="bf16",
             objective="sao", skip=False),
        # A trainer that upcasts its logits: float32 over the large vocabulary.
        dict(name="sapo_f32_151936", kind="fused", B=4, T=512, V=151936, dtype="f32",
             objective="sapo", skip=False),
        # GSPO: every log-prob of a sequence before any gradient.
        dict(name="gspo_bf16_151936", kind="fused", B=8, T=512, V=151936, dtype="bf16",
             objective="gspo", skip=False),
        # Scoring pass (old or reference log-probs), no gradient, through the
        # causal views logits[:, :-1], ids[:, 1:].
        dict(name="score_bf16_128256", kind="score", B=4, T=2048, V=128256, dtype="bf16"),
        # Supervised fine-tuning on an odd vocabulary.
        dict(name="sft_bf16_50257", kind="sft", B=8, T=1024, V=50257, dtype="bf16"),
        # From hidden states: LM head, log-probs, GRPO loss, both gradients.
        dict(name="lm_head_bf16", kind="linear", B=4, T=1024, V=151936, H=1024, dtype="bf16",
             objective="clipped"),
        # Advantages of a PPO batch: GAE, then whitening over its tokens.
        dict(name="gae_whiten_64x8192", kind="gae", B=64, T=8192, dtype="f32"),
        # One decode step of a rollout batch, the sampler's defaults.
        dict(name="sample_bf16_256", kind="sample", B=256, V=151936, dtype="bf16",
             setting="default"),
        # One decode step of a serving batch on float32 logits.
        dict(name="sample_f32_topk", kind="sample", B=64, V=151936, dtype="f32",
             setting="topk_topp"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng):
    if rng.random() < 0.5:
        return rng.choice([4096, 32000, 50257, 128256, 151936])
    return _log_uniform(rng, 2000, 160000)


def draw(rng):
    kind = rng.choice(["fused", "fused", "fused", "composed", "score", "sft", "linear", "gae",
                       "sample", "sample", "sample"])
    if kind == "gae":
        return dict(kind=kind, B=_log_uniform(rng, 8, 128), T=_log_uniform(rng, 64, 8192),
                    dtype="f32")
    V = _vocab(rng)
    if kind == "sample":
        return dict(kind=kind, B=_log_uniform(rng, 1, 256), V=V,
                    dtype=rng.choice(["bf16", "bf16", "f32", "f32", "f16"]),
                    setting=rng.choice(sorted(SETTINGS)))
    if kind == "linear":
        H = rng.choice([256, 512, 768, 1024, 2048])
        most = min(4096, int(4096 * 151936 * 1024 / (V * H)))
        tokens = _log_uniform(rng, 256, max(256, most))
        T = _log_uniform(rng, 16, max(16, tokens // GROUP))
        return dict(kind=kind, B=GROUP * max(1, tokens // (GROUP * T)), T=T, V=V, H=H,
                    dtype="bf16", objective=rng.choice(["clipped", "sapo"]))
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if kind == "score":
        dtype = rng.choice(["bf16", "bf16", "f32", "f16"])
    most = max(64, min(16384, int(4.0e9 / (V * SIZES[dtype]))))
    tokens = _log_uniform(rng, 64, most)
    T = _log_uniform(rng, 8, min(2048, max(8, tokens // GROUP)))
    B = GROUP * max(1, tokens // (GROUP * T))
    if kind == "score":
        return dict(kind=kind, B=B, T=T, V=V, dtype=dtype)
    if kind == "sft":
        return dict(kind=kind, B=B, T=T, V=V, dtype=dtype)
    case = dict(kind=kind, B=B, T=T, V=V, dtype=dtype, objective=rng.choice(sorted(OBJECTIVES)))
    if kind == "fused":
        case["skip"] = rng.random() < 0.2
    else:
        case["objective"] = "clipped"
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _logits(B, T, V, dtype, gen):
    """Logits ~ N(0, 3) with 5% of the rows carrying one dominant entry (+15),
    and actions sampled from their softmax (Gumbel-max)."""

    x = torch.empty(B, T, V, dtype=DTYPES[dtype], device=DEV)
    act = torch.empty(B, T, dtype=torch.int64, device=DEV)
    lp = torch.empty(B, T, dtype=torch.float32, device=DEV)
    rows = max(1, int(1.0e8) // V)
    flat, aflat, lflat = x.view(-1, V), act.view(-1), lp.view(-1)
    for r0 in range(0, B * T, rows):
        r1 = min(B * T, r0 + rows)
        z = torch.randn(r1 - r0, V, device=DEV, generator=gen) * 3.0
        hot = torch.rand(r1 - r0, device=DEV, generator=gen) < 0.05
        at = torch.randint(0, V, (r1 - r0, 1), device=DEV, generator=gen)
        z.scatter_add_(1, at, (15.0 * hot.float())[:, None])
        flat[r0:r1] = z.to(x.dtype)
        z = flat[r0:r1].float()
        u = torch.rand(r1 - r0, V, device=DEV, generator=gen).clamp_min_(1e-12)
        a = (z - torch.log(-torch.log(u))).argmax(dim=-1)
        aflat[r0:r1] = a
        lflat[r0:r1] = z.gather(1, a[:, None])[:, 0] - torch.logsumexp(z, dim=-1)
    return x, act, lp


def _mask(B, T, gen):
    n = torch.randint(max(1, T // 16), T + 1, (B, 1), device=DEV, generator=gen)
    return torch.arange(T, device=DEV)[None, :] < n


def _side(c, lp, gen):
    """Behaviour log-probs, per-sequence rewards and the action mask."""

    B, T = c["B"], c["T"]
    old = lp + 0.1 * torch.randn(B, T, device=DEV, generator=gen)
    rewards = torch.randn(B // GROUP, GROUP, device=DEV, generator=gen)
    return dict(old=old, rewards=rewards, mask=_mask(B, T, gen))


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + 17)
    c = dict(case)
    kind = c["kind"]
    s = dict(case=c)
    if kind == "gae":
        B, T = c["B"], c["T"]
        mask = _mask(B, T, gen)
        last = mask.sum(dim=1) - 1
        rewards = torch.zeros(B, T, device=DEV)
        rewards[torch.arange(B, device=DEV), last] = torch.randn(B, device=DEV, generator=gen)
        values = 0.5 * torch.randn(B, T, device=DEV, generator=gen)
        return dict(s, rewards=rewards, values=values, mask=mask)
    if kind == "sample":
        # next-token logits: a broad background under a few dozen candidates
        B, V = c["B"], c["V"]
        x = 1.5 * torch.randn(B, V, device=DEV, generator=gen)
        at = torch.randint(0, V, (B, 64), device=DEV, generator=gen)
        x.scatter_add_(1, at, 6.0 + 10.0 * torch.rand(B, 64, device=DEV, generator=gen))
        return dict(s, logits=x.to(DTYPES[c["dtype"]]), seed=int(seed) * 7919 + 11)
    if kind == "linear":
        B, T, V, H = c["B"], c["T"], c["V"], c["H"]
        h = torch.randn(B, T, H, device=DEV, generator=gen).to(DTYPES[c["dtype"]])
        w = (torch.randn(V, H, device=DEV, generator=gen) * (2.0 / math.sqrt(H))).to(h.dtype)
        act = torch.randint(0, V, (B, T), device=DEV, generator=gen)
        lp = torch.empty(B, T, device=DEV)
        for b in range(B):
            z = (h[b] @ w.t()).float()
            lp[b] = z.gather(1, act[b][:, None])[:, 0] - torch.logsumexp(z, dim=-1)
        s.update(_side(c, lp, gen))
        return dict(s, hidden=h.requires_grad_(), weight=w.requires_grad_(), act=act)
    x, act, lp = _logits(c["B"], c["T"], c["V"], c["dtype"], gen)
    if kind == "score":
        return dict(s, logits=x, act=act)
    if kind == "sft":
        labels = act.clone()
        labels[~_mask(c["B"], c["T"], gen)] = -100  # padding
        labels[:, 1:2] = act[:, 1:2]
        return dict(s, logits=x.requires_grad_(), labels=labels)
    s.update(_side(c, lp, gen))
    return dict(s, logits=x.requires_grad_(), act=act)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def _advantages(s):
    c = s["case"]
    adv = R.group_standardized_advantages(s["rewards"]).reshape(-1)
    if c["objective"] == "gspo":
        return adv
    return adv[:, None].expand(c["B"], c["T"])


def _scalars(out, objective):
    """The record's loss and diagnostics.  GSPO's sequence_ratio_divergence
    stays out: the mean of s - 1 - log s at s = 1 + O(1e-3) is a difference
    of float32 numbers near 1 and carries few digits by its nature."""

    if objective == "gspo":
        return [out.loss, out.sequence_clip_fraction, out.mean_sequence_ratio,
                out.sequence_ratios]
    if objective == "sao":
        return [out.loss, out.approximate_kl, out.rejected_fraction, out.mean_ratio,
                out.trusted_mask]
    if objective == "sapo":
        return [out.loss, out.approximate_kl, out.mean_ratio, out.mean_gradient_gate]
    return [out.loss, out.approximate_kl, out.clip_fraction, out.mean_ratio]


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "gae":
        adv, targets = R.generalized_advantage_estimation(
            s["rewards"], s["values"], gamma=1.0, gae_lambda=0.95, valid_mask=s["mask"])
        return dict(advantages=R.masked_whiten(adv, s["mask"]), targets=targets)
    if kind == "sample":
        temperature, top_k, top_p, do_sample, log_q = SETTINGS[c["setting"]]
        out = sample_next_token_batch(s["logits"], temperature, top_k, top_p, do_sample,
                                      seed=s["seed"], offset=3, sampling_logprobs=log_q)
        return dict(tokens=out.token_ids, logprobs=out.logprobs, q=out.sampling_logprobs)
    if kind == "score":
        with torch.no_grad():
            return R.gather_token_logprobs(s["logits"][:, :-1], s["act"][:, 1:])
    if kind == "sft":
        loss = causal_lm_loss(s["logits"], s["labels"])
        (dl,) = torch.autograd.grad(loss, s["logits"])
        return dict(loss=loss.detach(), dlogits=dl)
    obj = c["objective"]
    kw = OBJECTIVES[obj]
    if kind == "linear":
        out = R.fused_linear_policy_loss(s["hidden"], s["weight"], s["act"], s["old"],
                                         _advantages(s), s["mask"], objective=obj, **kw)
        dh, dw = torch.autograd.grad(out.loss, (s["hidden"], s["weight"]))
        return dict(scalars=[t.detach() for t in _scalars(out, obj)], dhidden=dh, dweight=dw)
    if kind == "composed":
        lp = R.gather_token_logprobs(s["logits"], s["act"])
        out = R.clipped_policy_loss(lp, s["old"], _advantages(s), s["mask"], **kw)
        (dl,) = torch.autograd.grad(out.loss, s["logits"])
        return dict(scalars=[t.detach() for t in _scalars(out, obj)], logprobs=lp.detach(),
                    dlogits=dl)
    out = R.fused_policy_loss(s["logits"], s["act"], s["old"], _advantages(s), s["mask"],
                              objective=obj, skip_masked_rows=c["skip"], **kw)
    (dl,) = torch.autograd.grad(out.loss, s["logits"])
    return dict(scalars=[t.detach() for t in _scalars(out, obj)], dlogits=dl)


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------


def work(case):
    c = case
    kind, B = c["kind"], c["B"]
    if kind == "gae":  # rewards, values, mask in; advantages, targets out
        return dict(bytes=B * c["T"] * (4 + 4 + 1 + 4 + 4), flops=0)
    if kind == "sample":
        return dict(bytes=B * c["V"] * SIZES[c["dtype"]] + 16 * B, flops=0)
    N, V, e = B * c["T"], c["V"], SIZES[c["dtype"]]
    if kind == "score":
        n = B * (c["T"] - 1)
        return dict(bytes=n * (V * e + 12), flops=0)
    if kind == "linear":  # logits, d hidden, d weight
        H = c["H"]
        return dict(bytes=2 * e * (N * H + V * H) + 21 * N, flops=6 * N * H * V)
    return dict(bytes=N * (2 * V * e + 21), flops=0)


def tolerance(case):
    kind = case["kind"]
    if kind == "gae":
        return dict(rel=1e-5, max=1e-3)
    if kind == "sample":
        # Without top-k and top-p a row's cumulative sums have V boundaries,
        # and sums in another order move a draw that lies on one to the next
        # token: 3 of 3072 rows between the package's two kernels (V = 151936),
        # none under the other settings.
        if case["setting"].startswith("default"):
            return dict(rel=0.03, max=0.9, differ=0.01)
        return dict(rel=2e-6, max=1e-4, differ=0.01)
    if kind == "score":
        return dict(rel=2e-6, max=1e-4)
    if kind == "linear":
        # the logits are rounded to bfloat16 before the softmax, as F.linear
        # leaves them: 1.6e-2 on either gradient against 64 bits
        return dict(rel=0.03, max=0.5)
    # bfloat16 gradients: half an ulp (2^-9) of rounding, 1.7e-3 in the
    # 2-norm.  The objectives' scalars are sums of terms of both signs.
    if case["dtype"] == "bf16":
        return dict(rel=6e-3, max=0.02, differ=1e-3)
    if kind == "fused" and case["objective"] == "gspo":
        return dict(rel=2e-3, max=0.02)
    return dict(rel=2e-5, max=1e-3, differ=1e-3)


# ---------------------------------------------------------------------------
# 64-bit results from plain torch
# ---------------------------------------------------------------------------


def _objective64(c, lp, old, adv, mask):
    """The objective (to be maximised) of float64 log-probs."""

    m = mask.double()
    kw = OBJECTIVES[c["objective"]]
    x = (lp - old).clamp(-20.0, 20.0)
    if c["objective"] == "gspo":
        s = (((lp - old) * m).sum(1) / m.sum(1)).clamp(-20.0, 20.0).exp()
        cl = s.clamp(1 - kw["clip_low"], 1 + kw["clip_high"])
        return torch.minimum(s * adv, cl * adv).mean()
    rho = x.exp()
    if c["objective"] == "clipped":
        cl = rho.clamp(1 - kw["clip_low"], 1 + kw["clip_high"])
        return (torch.minimum(rho * adv, cl * adv) * m).sum() / m.sum()
    if c["objective"] == "sao":
        w = rho.detach()
        trusted = (w > 1 - kw["clip_low"]) & (w < 1 + kw["clip_high"])
        return (torch.where(trusted, w * adv * lp, torch.zeros_like(lp)) * m).sum() / m.sum()
    tau = torch.where(adv > 0, kw["tau_positive"], kw["tau_negative"]).double()
    soft = (4.0 / tau) * torch.sigmoid(tau * (rho - 1.0)) * adv
    return ((soft * m).sum(1) / m.sum(1)).mean()


def _advantages64(s):
    c = s["case"]
    r = s["rewards"].double()
    d = r - r.mean(dim=1, keepdim=True)
    adv = (d / d.square().mean(dim=1, keepdim=True).sqrt()).reshape(-1)
    return adv if c["objective"] == "gspo" else adv[:, None].expand(c["B"], c["T"])


def _logprobs64(x, act):
    lp = torch.empty(act.shape, dtype=torch.float64, device=DEV)
    for b in range(x.shape[0]):
        z = x[b].double()
        lp[b] = z.gather(1, act[b][:, None])[:, 0] - torch.logsumexp(z, dim=-1)
    return lp


def _dlogits64(x, act, g):
    dl = torch.empty(x.shape, dtype=torch.float64, device=DEV)
    for b in range(x.shape[0]):
        torch.softmax(x[b].double(), dim=-1, out=dl[b])
        dl[b].mul_(-g[b][:, None])
        dl[b].scatter_add_(1, act[b][:, None], g[b][:, None])
    return dl


M32 = 0xFFFFFFFF


def _philox(ctr, key):
    """Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC 2011)."""

    c0, c1, c2, c3 = ctr
    k0, k1 = key
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c0, 0xCD9E8D57 * c2
        c0, c1, c2, c3 = (p1 >> 32) ^ c1 ^ k0, p1 & M32, (p0 >> 32) ^ c3 ^ k1, p0 & M32
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c0, c1, c2, c3


def _pick(w, u):
    """The first index whose cumulative weight exceeds u times the total."""

    cdf = torch.cumsum(w, 0)
    i = torch.searchsorted(cdf, (u * cdf[-1]).reshape(1), right=True)
    return i.clamp_max(w.numel() - 1)[0]


def _sample64(s):
    """The sampler's documented rule: the candidates of top-k and top-p (ties
    lowest index first) with weights max(p, 1e-9), drawn by inverse CDF in
    vocabulary order; without either, p and the floor's excess as a mixture."""

    temperature, top_k, top_p, do_sample, log_q = SETTINGS[s["case"]["setting"]]
    x = s["logits"].double()
    B, V = x.shape
    toks, lps, lqs = [], [], []
    for r in range(B):
        z = x[r] / (temperature if do_sample else 1.0)
        lse = torch.logsumexp(z, 0)
        if not do_sample:
            t, q = z.argmax(), z.new_zeros(())
        else:
            w = _philox((r, 0, 3, 0), (s["seed"] & M32, s["seed"] >> 32))
            u = (w[0] >> 8) * 2.0 ** -24
            u1 = (((w[1] << 21) | (w[2] >> 11)) & ((1 << 53) - 1)) * 2.0 ** -53
            order = torch.sort(z, descending=True, stable=True).indices
            cand = torch.ones(V, dtype=torch.bool, device=DEV)
            if 0 < top_k < V:
                cand.zero_()
                cand[order[:top_k]] = True
            p = torch.softmax(z.masked_fill(~cand, -math.inf), 0)
            if top_p < 1.0:
                drop = torch.cumsum(p[order], 0) > top_p
                drop[0] = False
                kept = torch.ones_like(cand)
                kept[order[drop]] = False
                wgt = (p * kept).clamp_min(1e-9) * cand
                t = _pick(wgt, u)
            elif 0 < top_k < V:
                wgt = p.clamp_min(1e-9) * cand
                t = _pick(wgt, u)
            else:
                g = (1e-9 - p).clamp_min(0.0)
                G = float(g.sum())
                wgt = p.clamp_min(1e-9)
                t = _pick(g if u1 < G / (1.0 + G) else p, u)
            q = torch.log(wgt[t] / wgt.sum())
        toks.append(t)
        lps.append(z[t] - lse)
        lqs.append(q)
    return dict(tokens=torch.stack(toks), logprobs=torch.stack(lps),
                q=torch.stack(lqs) if log_q else None)


def exact(case, seed):
    s = prepare(case, seed)
    c = s["case"]
    kind = c["kind"]
    with torch.no_grad():
        if kind == "sample":
            return _sample64(s)
        if kind == "score":
            return _logprobs64(s["logits"][:, :-1], s["act"][:, 1:])
        if kind == "gae":
            m = s["mask"]
            r, v = s["rewards"].double(), s["values"].double()
            adv, tgt = torch.zeros_like(r), torch.zeros_like(r)
            nv, na = torch.zeros_like(r[:, 0]), torch.zeros_like(r[:, 0])
            for t in range(c["T"] - 1, -1, -1):
                a = r[:, t] + nv - v[:, t] + 0.95 * na
                nv, na = torch.where(m[:, t], v[:, t], nv), torch.where(m[:, t], a, na)
                adv[:, t] = torch.where(m[:, t], a, torch.zeros_like(a))
                tgt[:, t] = torch.where(m[:, t], a + v[:, t], torch.zeros_like(a))
            x = adv[m]
            out = (adv - x.mean()) / (x.var(unbiased=False).sqrt() + 1e-8)
            return dict(advantages=torch.where(m, out, torch.zeros_like(out)), targets=tgt)
        if kind == "sft":
            x, lab = s["logits"].detach(), s["labels"][:, 1:]
            live = lab != -100
            tgt = torch.where(live, lab, torch.zeros_like(lab))
            lp = _logprobs64(x[:, :-1], tgt)
            g = -live.double() / live.sum()
            dl = torch.zeros(x.shape, dtype=torch.float64, device=DEV)
            dl[:, :-1] = _dlogits64(x[:, :-1], tgt, g)
            return dict(loss=-(lp * live).sum() / live.sum(), dlogits=dl)
        if kind == "linear":
            h = s["hidden"].detach().double().reshape(-1, c["H"])
            w = s["weight"].detach().double()
            x = (h @ w.t()).view(c["B"], c["T"], c["V"])
        else:
            x = s["logits"].detach()
        lp = _logprobs64(x, s["act"])
    lp.requires_grad_()
    loss = -_objective64(c, lp, s["old"].double(), _advantages64(s), s["mask"])
    (g,) = torch.autograd.grad(loss, lp)
    # The scalars are sums of terms of both signs that nearly cancel: their
    # relative error in 32 bits says nothing, so no 64-bit value stands here.
    n = dict(gspo=4, sao=5).get(c["objective"], 4)
    with torch.no_grad():
        dl = _dlogits64(x, s["act"], g)
        if kind == "linear":
            d2 = dl.view(-1, c["V"])
            return dict(scalars=[None] * n, dhidden=(d2 @ w).view(s["hidden"].shape),
                        dweight=d2.t() @ h)
    out = dict(scalars=[None] * n, dlogits=dl)
    if kind == "composed":
        out["logprobs"] = lp.detach()
    return out
