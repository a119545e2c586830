"""Attention on bf16 pieces (attention_x3.hip): tile edges of queries, keys and
head dims, both query splits, masks and weights, and the values the pieces
cannot carry.

Bar against float64: a score is within e = scale (d / 32 + 12) 2^-24 |q||k| of
the exact one (the products' rounding, as in the GEMM on pieces) plus 2^-23 of
itself (scale, the exponent's product), so a weight is within a factor
1 + 2 max e + (skv / 32 + 32) 2^-24 (its sum, the exponential, the division)
and an output within that plus 6 roundings per 32 keys of the sum over
w |v|.  Terms below 2^-126 may be flushed."""
import math

import pytest

pytestmark = pytest.mark.gpu


def _gh():
    import ghostflow_hip
    return ghostflow_hip


def _kept(torch, b, h, sq, skv, causal, mask, dev):
    keep = torch.ones(b, h, sq, skv, dtype=torch.bool, device=dev)
    if causal:
        keep &= torch.ones(sq, skv, dtype=torch.bool, device=dev).tril(skv - sq)
    if mask is not None:
        flat = torch.arange(b * h * sq * skv, device=dev) % mask.numel()
        keep &= (mask.reshape(-1)[flat] > 0.5).reshape(b, h, sq, skv)
    return keep


def _reference(torch, q, k, v, keep, scale):
    """Output, weights, and the bars of both, in float64."""
    q, k, v = q.double(), k.double(), v.double()
    d, skv = q.shape[-1], k.shape[-2]
    kt = k.transpose(-1, -2).contiguous()
    s = (q @ kt) * scale
    e = (q.abs() @ kt.abs()) * (scale * (d / 32 + 12) * 2.0 ** -24) + s.abs() * 2.0 ** -23
    s = s.masked_fill(~keep, -math.inf)
    w = torch.softmax(s, -1)
    rel = 2 * torch.where(keep, e, 0).amax(-1, keepdim=True) + (skv / 32 + 32) * 2.0 ** -24
    wv = w @ v.abs()
    return w @ v, w, wv * (rel + 6 * skv / 32 * 2.0 ** -24) + skv * 2.0 ** -126, w * rel + 2.0 ** -125


def _mask(torch, kind, sq, skv, g, dev):
    if kind == "none":
        return None
    if kind == "tril":  # one mask for every (batch, head); whole tiles masked
        return torch.ones(sq, skv, device=dev).tril(skv - sq)
    m = (torch.rand(2 * skv + 7 if kind == "odd" else 3 * skv, device=dev, generator=g) > 0.3).float()
    m[::3 if kind == "odd" and skv > 2 else 1 if kind == "odd" else skv] = 1.0  # every row keeps a key
    return m


def _check(torch, dev, b, h, sq, skv, d, causal, kind, weights, seed=0, tweak=None):
    gh = _gh()
    g = torch.Generator(device=dev)
    g.manual_seed(seed + sq * 7 + skv * 3 + d)
    q = torch.randn(b, h, sq, d, device=dev, generator=g)
    k = torch.randn(b, h, skv, d, device=dev, generator=g)
    v = torch.randn(b, h, skv, d, device=dev, generator=g)
    mask = _mask(torch, kind, sq, skv, g, dev)
    if tweak:
        tweak(q, k, v)
    keep = _kept(torch, b, h, sq, skv, causal, mask, dev)
    assert keep.any(-1).all()
    ref, rw, bar, wbar = _reference(torch, q, k, v, keep, 1.0 / math.sqrt(d))
    got = gh.sdpa(q, k, v, causal=causal, mask=mask, want_weights=weights)
    if weights:
        got, w = got
        assert ((w.double() - rw).abs() <= wbar).all(), float(((w.double() - rw).abs() / wbar).max())
        assert (w[~keep] == 0).all()
    assert ((got.double() - ref).abs() <= bar).all(), float(((got.double() - ref).abs() / bar).max())


@pytest.mark.parametrize("d", [4, 20, 32, 36, 64, 68, 96, 100, 128])
@pytest.mark.parametrize("sq,skv", [(1, 1), (16, 31), (17, 33), (128, 64), (129, 257), (300, 95)])
def test_edges(torch_dev, sq, skv, d):
    import torch
    n = min(sq, skv)
    _check(torch, torch_dev, 1, 3, n, n, d, True, "none", False)
    _check(torch, torch_dev, 2, 1, sq, skv, d, False, "none", False)
    _check(torch, torch_dev, 1, 2, sq, skv, d, False, "odd", True)


@pytest.mark.parametrize("d", [64, 80, 128])
@pytest.mark.parametrize("kind", ["tril", "rows"])
@pytest.mark.parametrize("s", [36, 130, 260])
def test_masks_and_weights(torch_dev, s, kind, d):
    import torch
    for weights in (False, True):
        _check(torch, torch_dev, 2, 3, s, s, d, False, kind, weights)
        _check(torch, torch_dev, 1, 3, s, s, d, True, kind, weights)


@pytest.mark.parametrize("d", [72, 128])
@pytest.mark.parametrize("causal,kind", [(True, "none"), (False, "none"), (False, "tril"), (True, "rows")])
def test_two_sets_per_wave(torch_dev, d, causal, kind):
    """Launches of at least 512 blocks of 256 queries, with a partial one."""
    import torch
    _check(torch, torch_dev, 4, 43, 530, 530, d, causal, kind, False)


@pytest.mark.parametrize("d", [72, 96, 128])
@pytest.mark.parametrize("sq,skv", [(1, 1), (1, 300), (16, 33), (17, 95), (64, 130), (65, 64)])
def test_few_queries_many_slices(torch_dev, sq, skv, d):
    """More slices than CUs: up to 64 queries run on workgroups of four waves."""
    import torch
    _check(torch, torch_dev, 2, 131, sq, skv, d, False, "none", False)
    _check(torch, torch_dev, 2, 131, sq, skv, d, False, "odd", True)
    _check(torch, torch_dev, 131, 2, sq, sq, d, True, "none", sq % 2 == 0)


@pytest.mark.parametrize("d", [20, 64, 128])
def test_wide_ranges(torch_dev, d):
    """Large logits, small and large values, and elements beyond the pieces
    that the exact result can carry."""
    import torch

    def logits(q, k, v):
        q.mul_(30.0)

    def small(q, k, v):
        v.mul_(1e-33)

    def large(q, k, v):
        v.mul_(1e25)

    def mixed(q, k, v):
        q.mul_(1e-22)
        k.mul_(1e22)

    for t in (logits, small, large, mixed):
        _check(torch, torch_dev, 1, 2, 70, 100, d, False, "odd", True, tweak=t)
        _check(torch, torch_dev, 1, 2, 100, 100, d, True, "none", False, tweak=t)


def test_non_finite_values(torch_dev):
    """A query's infinity or NaN stays in its row; one in V reaches every
    query, also through a masked weight of 0; one in a masked key reaches
    none; a row with nothing kept is NaN."""
    import torch
    gh = _gh()
    q, k, v = (torch.randn(1, 2, 150, 64, device=torch_dev) for _ in range(3))
    mask = torch.ones(150, 150, device=torch_dev).tril()
    clean, cw = gh.sdpa(q, k, v, mask=mask, want_weights=True)
    for bad in (math.inf, math.nan):
        q2 = q.clone()
        q2[0, 0, 5, 3] = bad
        o, w = gh.sdpa(q2, k, v, mask=mask, want_weights=True)
        assert o[0, 0, 5].isnan().all() and w[0, 0, 5, :6].isnan().all()
        o[0, 0, 5], w[0, 0, 5] = clean[0, 0, 5], cw[0, 0, 5]
        torch.testing.assert_close(o, clean, rtol=0, atol=1e-5)
        torch.testing.assert_close(w, cw, rtol=0, atol=1e-5)
        v2 = v.clone()
        v2[0, 1, 149, 7] = bad
        o = gh.sdpa(q, k, v2, mask=mask)
        assert o[0, 1, :149, 7].isnan().all() and not o[0, 1, 149, 7].isfinite()
        o[0, 1, :, 7] = clean[0, 1, :, 7]
        torch.testing.assert_close(o, clean, rtol=0, atol=1e-5)
        k2 = k.clone()
        k2[0, 0, 149] = bad
        o = gh.sdpa(q, k2, v, mask=mask)
        torch.testing.assert_close(o[:, :, :149], clean[:, :, :149], rtol=0, atol=1e-5)
    mask[40] = 0.0
    o, w = gh.sdpa(q, k, v, mask=mask, want_weights=True)
    assert o[:, :, 40].isnan().all() and w[:, :, 40].isnan().all()
    assert o[:, :, :40].isfinite().all() and o[:, :, 41:].isfinite().all()


def test_out_may_be_q(torch_dev):
    import torch
    gh = _gh()
    for scale in (1.0, 1e25):  # on pieces; on the f32 units
        q, k, v = (torch.randn(1, 3, 200, 96, device=torch_dev) for _ in range(3))
        v *= scale
        ref = gh.sdpa(q, k, v, causal=True)
        gh.sdpa(q, k, v, causal=True, out=q)
        assert torch.equal(q, ref)


def test_many_slices(torch_dev):
    """2^23 (batch, head) slices: beyond the grid of the kernel on pieces."""
    import torch
    gh = _gh()
    b, h = 1 << 12, 1 << 11
    q, k, v = (torch.randn(b, h, 1, 4, device=torch_dev) for _ in range(3))
    assert torch.equal(gh.sdpa(q, k, v), v)


@pytest.mark.parametrize("d", [20, 64, 128])
@pytest.mark.parametrize("weights", [False, True])
def test_nan_scores_reach_their_rows(torch_dev, weights, d):
    """A kept NaN score makes its whole row NaN (the reference's maximum ignores
    it, the sum of the row does not), also where every score before it, or the
    whole first key tile, is NaN; a masked one leaves its row alone."""
    import torch
    gh = _gh()
    s = 70
    q, k, v = (torch.randn(1, 2, s, d, device=torch_dev) for _ in range(3))

    def run(kk, **kw):
        r = gh.sdpa(q, kk, v, want_weights=weights, **kw)
        return r if weights else (r, r)

    for first in (16, 32, 40):
        bad = k.clone()
        bad[0, 0, :first] = math.nan
        for causal in (False, True):
            clean = run(k, causal=causal)
            for x, c in zip(run(bad, causal=causal), clean):
                assert x[0, 0].isnan().all()
                torch.testing.assert_close(x[0, 1], c[0, 1], rtol=0, atol=1e-5)
    # of the first 16 keys, rows 10 .. 19 keep the NaN one alone and rows
    # 20 .. 29 none of the NaN ones
    bad = k.clone()
    bad[0, 0, 3] = math.nan
    mask = torch.ones(s, s, device=torch_dev)
    mask[10:20, :16] = 0.0
    mask[10:20, 3] = 1.0
    mask[20:30, 3] = 0.0
    rows = torch.zeros(s, dtype=torch.bool, device=torch_dev)
    rows[20:30] = True
    for x, c in zip(run(bad, mask=mask), run(k, mask=mask)):
        assert x[0, 0, ~rows].isnan().all()
        torch.testing.assert_close(x[0, 0, rows], c[0, 0, rows], rtol=0, atol=1e-5)


def test_nan_scores_many_slices(torch_dev):
    """The same in the kernel for 2^23 and more (batch, head) slices."""
    import torch
    gh = _gh()
    b, h, skv, d = 1 << 12, 1 << 11, 40, 4
    q, k, v = (torch.empty(b, h, n, d, device=torch_dev).normal_() for n in (1, skv, skv))
    k[7, 9, :32] = math.nan
    for weights in (False, True):
        r = gh.sdpa(q, k, v, want_weights=weights)
        for x in r if weights else (r,):
            assert x[7, 9].isnan().all()
            assert x[7, 8].isfinite().all() and x[7, 10].isfinite().all()


@pytest.mark.parametrize("d", [4, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_small_weights_and_values(torch_dev, causal, d):
    """A weight of 2^-124 keeps fp32 precision where V is zero at the larger
    ones, and V down to the subnormals keeps its bits.  Scores are exact here
    (one product of small integers each), so a weight is within |s| 2^-23 (the
    exponent's product) + 2^-19 (the rounded exponent of up to 2^7, times
    ln 2) + 8 2^-24, and the output 8 2^-24 more."""
    import torch
    gh = _gh()
    s = 40
    q, k = torch.zeros(1, 2, s, d, device=torch_dev), torch.zeros(1, 2, s, d, device=torch_dev)
    q[..., 0] = 2.0
    k[..., 0] = -86.0
    k[:, :, 0, 0] = 0.0
    scale = 0.5
    g = torch.Generator(device=torch_dev).manual_seed(d)
    for e in (50, 0, -20):
        v = torch.randn(1, 2, s, d, device=torch_dev, generator=g) * 2.0 ** e
        v[:, :, 0] = 0.0
        got = gh.sdpa(q, k, v, scale=scale, causal=causal)
        x = (q.double() @ k.double().transpose(-1, -2).contiguous()) * scale
        if causal:
            x = x.masked_fill(~torch.ones(s, s, dtype=torch.bool, device=torch_dev).tril(), -math.inf)
        w = torch.softmax(x, -1)
        ref, bar = w @ v.double(), w @ v.double().abs()
        # (fp32 weights and outputs below 2^-126 round to 2^-149)
        assert ((got.double() - ref).abs() <= bar * (86 * 2.0 ** -23 + 2.0 ** -19 + 16 * 2.0 ** -24) + s * 2.0 ** -148).all(), \
            (e, float(((got.double() - ref).abs() / bar.clamp_min(1e-300)).max()))
    # subnormal values under ordinary weights
    q, k = (torch.randn(1, 2, s, d, device=torch_dev, generator=g) for _ in range(2))
    for e in (-118, -130, -140):
        v64 = torch.randn(1, 2, s, d, device=torch_dev, generator=g).double() * 2.0 ** e
        v = v64.float()
        got = gh.sdpa(q, k, v, causal=causal)
        keep = _kept(torch, 1, 2, s, s, causal, None, torch_dev)
        ref, _, bar, _ = _reference(torch, q, k, v, keep, 1.0 / math.sqrt(d))
        assert ((got.double() - ref).abs() <= bar - s * 2.0 ** -126 + 2.0 ** -148).all(), e
