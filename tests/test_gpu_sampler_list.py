"""The streaming sampler's candidate lists (MI355X): top-k and top-p from the
lane maxima, at the sizes where the list fits, overflows or ends before the
nucleus does, against the CPU oracle; and a draw that falls on the floor
entries between the kept ones.

A row is decided when its uniform lies more than 1e-5 of the total from a
cumulative boundary and top_p more than 1e-6 from the nucleus cut, as in
test_gpu_sampler.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import sampler_oracle as so
from rosellm_amd import roseinfer as RI

pytestmark = pytest.mark.gpu


def _rows(kind, B, V, dtype):
    g = torch.Generator().manual_seed(V + B)
    x = torch.randn(B, V, generator=g)
    if kind == "peaked":
        x[:, ::97] += 6.0
    elif kind == "flat":  # the nucleus reaches past any list
        x *= 0.01
    elif kind == "ties":  # a few values: thresholds are large tie groups
        x = torch.round(2.0 * x)
    elif kind == "masked":  # fewer finite entries than lanes
        x[torch.rand(B, V, generator=g) < 1.0 - 90.0 / V] = -float("inf")
        x[:, V // 2] = 1.0
    elif kind == "clump":  # the candidates share lanes
        x[:, V // 3:V // 3 + 40] += 7.0
    return x.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("V", [5, 63, 1025, 4099, 9001, 50257])
@pytest.mark.parametrize("kind", ["peaked", "flat", "ties"])
@pytest.mark.parametrize("top_k,top_p", [(1, 1.0), (40, 0.9), (64, 1.0), (300, 0.95), (0, 0.9),
                                         (0, 0.3)])
def test_lists(device, dtype, V, kind, top_k, top_p):
    print(f"[sampler list] {dtype} V={V} {kind} k={top_k} p={top_p}", flush=True)
    B = 6
    x = _rows(kind, B, V, dtype)
    wide = torch.zeros(B, V + 3, dtype=dtype, device=device)
    wide[:, 1:V + 1] = x.to(device)  # rows off every 16-byte boundary
    kw = dict(temperature=0.8, top_k=top_k, top_p=top_p, do_sample=True)
    want = so.sample_rows(x.float().numpy(), seed=7, offset=2, **kw)
    for rows in (x.to(device), wide[:, 1:V + 1]):
        out = RI.sample_next_token_batch(rows, seed=7, offset=2, **kw)
        sure = torch.from_numpy((want["margin"] > 1e-5) & (want["p_margin"] > 1e-6))
        tok = torch.from_numpy(want["token"])
        assert torch.equal(out.token_ids.cpu()[sure], tok[sure])
        for got, w in ((out.logprobs, want["logp"]), (out.sampling_logprobs, want["logq"])):
            w = torch.from_numpy(w)[sure]
            assert torch.allclose(got.cpu().double()[sure], w, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("kind", ["peaked", "masked", "clump"])
@pytest.mark.parametrize("kb", [12, 24, 48])
@pytest.mark.parametrize("side", [-1, 1])
def test_list_or_passes(device, kind, kb, side):
    """Row lengths on both sides of the top-k list's limits, at each limit and one
    past it, and nuclei that end inside and beyond the list."""

    for dtype, size in ((torch.float32, 4), (torch.float16, 2)):
        V = (kb << 10) // size + side
        print(f"[sampler list] {dtype} V={V} {kind}", flush=True)
        x = _rows(kind, 4, V, dtype)
        for top_k, top_p in [(50, 1.0), (51, 0.9), (300, 1.0), (301, 1.0), (400, 0.95), (401, 1.0),
                             (600, 1.0), (601, 1.0), (0, 0.5), (0, 0.8), (0, 0.97)]:
            kw = dict(temperature=0.8, top_k=top_k, top_p=top_p, do_sample=True)
            want = so.sample_rows(x.float().numpy(), seed=7, offset=2, **kw)
            out = RI.sample_next_token_batch(x.to(device), seed=7, offset=2, **kw)
            sure = torch.from_numpy((want["margin"] > 1e-5) & (want["p_margin"] > 1e-6))
            assert torch.equal(out.token_ids.cpu()[sure], torch.from_numpy(want["token"])[sure])
            for got, w in ((out.logprobs, want["logp"]), (out.sampling_logprobs, want["logq"])):
                w = torch.from_numpy(w)[sure]
                assert torch.allclose(got.cpu().double()[sure], w, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_draw_on_the_floor(device, dtype):
    """Two kept entries in the middle of 151,936: the other entries' floor of
    1e-9 each is 1.5e-4 of the total, about ten of 65,536 draws.  The kept
    weights carry float32 rounding, 2^-23 of the total or 120 floors each, so a
    floor token may sit that far from the exact one."""

    V, B = 151936, 65536
    x = torch.full((1, V), -30.0)
    x[0, 60000], x[0, 110000] = 3.0, 2.5
    x = x.to(dtype)
    out = RI.sample_next_token_batch(x.to(device).expand(B, V), 1.0, 0, 0.95, True, seed=3,
                                     offset=1)
    tok = out.token_ids.cpu().numpy()
    q, _ = so.sampling_distribution(x.float().numpy()[0].astype(np.float64), 1.0, 0, 0.95)
    cdf = np.cumsum(q)
    u = np.array([so.row_uniform(3, 1, r) for r in range(B)])
    want = np.searchsorted(cdf, u * cdf[-1], side="right")
    kept = np.isin(want, np.nonzero(q > 1e-8)[0])
    assert 3 <= (~kept).sum() <= 40
    near = np.minimum(np.abs(cdf[want] - u * cdf[-1]),
                      np.abs(u * cdf[-1] - (cdf[want] - q[want]))) < 1e-6
    assert (tok[kept & ~near] == want[kept & ~near]).all()
    assert (np.abs(tok[~kept] - want[~kept]) <= 300).all()
    floor = torch.from_numpy(~np.isin(tok, np.nonzero(q > 1e-8)[0]))
    lq = out.sampling_logprobs.cpu().double()[floor]
    assert torch.allclose(lq, torch.full_like(lq, float(np.log(1e-9 / cdf[-1]))), atol=1e-4)
