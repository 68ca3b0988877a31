"""The reverse scans and the masked whitening at the edges of their tiles
(MI355X), against a plain walk through time in float64.

Sequence lengths sit on, and one past, one wave (256 steps), one 256-lane
tile (1024) and one and two 1024-lane tiles (8192, 16384); lengths that are
not multiples of four and strided operands take the element-wise loads.  Bars:
the carried state is a sum of at most T terms in float32 (1e-5 of the largest
term); whitening 1e-5 relative.
"""

from __future__ import annotations

import pytest
import torch

from rosellm_amd import roserlhf as R

pytestmark = pytest.mark.gpu

LENGTHS = [1, 3, 4, 255, 256, 257, 260, 1023, 1024, 1025, 1028, 8191, 8192, 8196, 16384, 16388]


def _inputs(B, T, device):
    g = torch.Generator(device=device).manual_seed(T)
    r = torch.randn(B, T, device=device, generator=g)
    v = torch.randn(B, T, device=device, generator=g)
    nv = torch.randn(B, T, device=device, generator=g)
    valid = torch.rand(B, T, device=device, generator=g) < 0.8
    term = torch.rand(B, T, device=device, generator=g) < 0.01
    valid[0, -1] = False
    if B > 2:
        valid[2] = False  # nothing but padding
    boot = torch.randn(B, device=device, generator=g)
    return r, v, nv, valid, term, boot


def _walk(r, v, nv, valid, term, boot, gamma, lam):
    r, v, nv, boot = (x.double().cpu() for x in (r, v, nv, boot))
    ok, nt = valid.cpu(), (~term.cpu()).double()
    B, T = r.shape
    ret, gae, tgt, skip = (torch.zeros(B, T, dtype=torch.float64) for _ in range(4))
    R0, V1, A1, A2 = boot.clone(), boot.clone(), torch.zeros(B).double(), torch.zeros(B).double()
    for t in range(T - 1, -1, -1):
        m = ok[:, t]
        R0 = torch.where(m, r[:, t] + gamma * nt[:, t] * R0, R0)
        ret[:, t] = torch.where(m, R0, 0.0)
        a = r[:, t] + gamma * nt[:, t] * V1 - v[:, t] + gamma * lam * nt[:, t] * A1
        A1, V1 = torch.where(m, a, A1), torch.where(m, v[:, t], V1)
        gae[:, t] = torch.where(m, a, 0.0)
        tgt[:, t] = torch.where(m, a + v[:, t], 0.0)
        a = r[:, t] + gamma * nt[:, t] * nv[:, t] - v[:, t] + gamma * lam * nt[:, t] * A2
        A2 = torch.where(m, a, A2)
        skip[:, t] = torch.where(m, a, 0.0)
    return ret, gae, tgt, skip


def _near(got, want):
    scale = max(1.0, want.abs().max().item())
    assert (got.double().cpu() - want).abs().max().item() <= 1e-5 * scale


@pytest.mark.parametrize("T", LENGTHS)
@pytest.mark.parametrize("strided", [False, True])
def test_scans(device, T, strided):
    print(f"[scan] T={T} strided={strided}", flush=True)
    ins = _inputs(3, T, device)
    if strided:  # every second element of a wider tensor
        wide = lambda x: torch.stack([x, torch.zeros_like(x)], -1).reshape(3, -1)[:, ::2]  # noqa: E731
        ins = tuple(wide(x) if x.ndim == 2 else x for x in ins)
    r, v, nv, valid, term, boot = ins
    ret, gae, tgt, skip = _walk(*ins, 0.99, 0.95)
    kw = dict(terminated=term, valid_mask=valid)
    _near(R.discounted_returns(r, gamma=0.99, bootstrap_value=boot, **kw), ret)
    a, t = R.generalized_advantage_estimation(r, v, gamma=0.99, gae_lambda=0.95,
                                              bootstrap_value=boot, **kw)
    _near(a, gae)
    _near(t, tgt)
    a, _ = R.skip_observation_generalized_advantage_estimation(r, v, nv, gamma=0.99,
                                                               gae_lambda=0.95, **kw)
    _near(a, skip)


def test_gae_infinite_value_stays_where_the_recurrence_has_it(device):
    """An infinite value reaches its own step and, through the bootstrap and
    the trace, the steps before it; a terminal step's products with zero make
    NaN as the reference's do."""

    r, v, nv, valid, term, boot = _inputs(2, 512, device)
    valid[:], term[:] = True, False
    v[0, 300] = float("inf")
    ins = (r, v, nv, valid, term, boot)
    _, gae, tgt, _ = _walk(*ins, 1.0, 0.0)
    a, t = R.generalized_advantage_estimation(r, v, gamma=1.0, gae_lambda=0.0,
                                              bootstrap_value=boot)
    assert torch.equal(torch.isnan(a.cpu()), torch.isnan(gae))
    assert torch.equal(torch.isinf(t.cpu()), torch.isinf(tgt))


@pytest.mark.parametrize("B,T", [(1, 1), (1, 2047), (1, 2048), (3, 683), (7, 4099), (1, 2100000)])
@pytest.mark.parametrize("layout", ["flat", "offset", "strided"])
def test_whiten_tiles(device, B, T, layout):
    """One tile of 2048 elements, a remainder, and more tiles than workgroups;
    a large common offset, which a one-pass sum of squares would lose."""

    g = torch.Generator(device=device).manual_seed(T)
    x = 1000.0 + torch.randn(B, T, device=device, generator=g)
    m = torch.rand(B, T, device=device, generator=g) < 0.6
    m[0, 0] = True
    if layout == "strided":
        x = torch.stack([x, x], -1).reshape(B, -1)[:, ::2]
    elif layout == "offset":  # contiguous, but not at a 16-byte address
        x = torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(B, T)
    xd = x.double()[m]
    sd = xd.var(unbiased=False).sqrt() if xd.numel() > 1 else xd.new_zeros(())
    want = torch.where(m, (x.double() - xd.mean()) / (sd + 1e-3), 0.0)
    got = R.masked_whiten(x, m, eps=1e-3)
    # float32 mean of values near 1000: 1e-4 of a standard deviation
    assert (got.double() - want).abs().max().item() <= 1e-3 * max(1.0, want.abs().max().item())
    with pytest.raises(ValueError):
        R.masked_whiten(x, torch.zeros_like(m))


@pytest.mark.parametrize("layout", ["flat", "strided"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_whiten_large_values(device, layout, dtype):
    """Finite values whose squares overflow float32 while their deviations do
    not, in one tile of 2048 elements and in several."""

    def run(x, m):
        if layout == "strided":
            x = torch.stack([x, x], -1).reshape(x.shape[0], -1)[:, ::2]
        return R.masked_whiten(x, m).double()

    for n in (64, 4096):
        m = torch.ones(1, n, dtype=torch.bool, device=device)
        # deviations of 1e17 about 2e19
        x = (2.0e19 + 1.0e17 * torch.randn(1, n, device=device)).to(dtype)
        xd = x.double()
        want = (xd - xd.mean()) / xd.var(unbiased=False).sqrt()
        # float32 mean: 1e-6 of 2e19, 2e-4 of a deviation; bfloat16 results are
        # rounded to 8 bits, 2^-9 of a value at most
        bar = 1e-3 + (2.0 ** -9 if dtype == torch.bfloat16 else 0.0)
        assert (run(x, m) - want).abs().max().item() <= bar * want.abs().max().item()
        # one value 2^n times: its sum is exact, so nothing deviates
        x = torch.full((1, n), 2.0 ** 100, dtype=dtype, device=device)
        assert torch.equal(run(x, m), torch.zeros(1, n, dtype=torch.float64, device=device))
    # two tiles with one value each: the means lie two deviations apart
    m = torch.zeros(1, 4096, dtype=torch.bool, device=device)
    m[0, 5] = m[0, 3000] = True
    x = torch.zeros(1, 4096, dtype=dtype, device=device)
    x[0, 5], x[0, 3000] = 2.0 ** 63.5, -(2.0 ** 63.5)
    got = run(x, m)
    assert abs(got[0, 5].item() - 1.0) <= 1e-2 and got[0, 3000].item() == -got[0, 5].item()
    # a spread whose square no float32 holds: deviations over an infinite one
    x[0, 5], x[0, 3000] = 3.0e38, -3.0e38
    assert torch.equal(run(x, m), torch.zeros_like(got))
