"""Prompt attention (`miq_attention`) against float64 at the edges of its tiles: fewer rows than a
tile, one row more, a cache that starts part way, key counts around a block and around the four
waves' share, the last position of the cache; and NaN or infinite value rows, which reach exactly
the queries that attend to them."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(q, k, v, pos):
    import torch
    from webpytorch_amd import _lib, core
    T, NH, HD = q.shape
    NKV, LMAX = k.shape[:2]
    st = torch.zeros(_lib.lib().miq_decode_state_words(), dtype=torch.int32, device="cuda")
    st[0] = pos
    out = torch.full_like(q, 7.0)
    _lib.call("miq_attention", core.ptr(q), core.ptr(k), core.ptr(v), core.ptr(st), core.ptr(out), T, NH, NKV, HD,
              LMAX, 1.0 / math.sqrt(HD), core.stream_handle())
    return out


def want(q, k, v, pos):
    import torch
    T, NH, HD = q.shape
    rep, LMAX = NH // k.shape[0], k.shape[1]
    out = torch.empty(T, NH, HD, dtype=torch.float64)
    for t in range(T):
        S = min(pos + t + 1, LMAX)
        for h in range(NH):
            s = (k[h // rep, :S].double() @ q[t, h].double()) / math.sqrt(HD)
            out[t, h] = torch.softmax(s, 0) @ v[h // rep, :S].double()
    return out


@pytest.mark.parametrize("NH,NKV,HD", [(4, 2, 64), (3, 1, 128), (2, 2, 32)])
@pytest.mark.parametrize("T,pos,LMAX", [(1, 0, 1), (1, 31, 64), (15, 0, 16), (17, 0, 40), (33, 127, 160), (16, 112, 128),
                                        (5, 500, 505), (130, 3, 140)])
def test_attention_matches_float64(gpu, NH, NKV, HD, T, pos, LMAX):
    import torch
    g = torch.Generator().manual_seed(T * 1000 + pos + HD)
    q, k, v = (torch.randn(s, generator=g) for s in ((T, NH, HD), (NKV, LMAX, HD), (NKV, LMAX, HD)))
    got = run(q.cuda(), k.cuda(), v.cuda(), pos).cpu().double()
    ref = want(q, k, v, pos)
    # scores carry HD roundings of 2^-24 at |s| <= ~5, so p is within ~1e-6 relatively at worst
    assert float((got - ref).norm() / ref.norm()) < 2e-6
    assert float((got - ref).abs().max()) < 2e-5


@pytest.mark.parametrize("HD", [64, 128])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_non_finite_values_reach_only_their_queries(gpu, HD, bad):
    """A value row of position 20 and stale rows past the last position: queries before position
    20 are what they are without them, later ones are non-finite in that dimension only."""
    import torch
    g = torch.Generator().manual_seed(HD)
    T, NH, LMAX = 40, 2, 96
    q, k, v = (torch.randn(s, generator=g) for s in ((T, NH, HD), (1, LMAX, HD), (1, LMAX, HD)))
    clean = run(q.cuda(), k.cuda(), v.cuda(), 0).cpu()
    v[0, 20, 5] = bad
    v[0, T:] = bad
    k[0, T:] = bad
    got = run(q.cuda(), k.cuda(), v.cuda(), 0).cpu()
    np.testing.assert_allclose(got[:20].numpy(), clean[:20].numpy(), rtol=0, atol=1e-5)
    other = torch.arange(HD) != 5
    np.testing.assert_allclose(got[20:][..., other].numpy(), clean[20:][..., other].numpy(), rtol=0, atol=1e-5)
    assert not torch.isfinite(got[20:, :, 5]).any()


@pytest.mark.parametrize("NH,NKV,HD", [(2, 1, 64), (2, 1, 128), (2, 1, 32)])
@pytest.mark.parametrize("big", [1e36, 2e38])
def test_values_near_the_fp32_range(gpu, NH, NKV, HD, big):
    """Values whose sum over the keys is past the fp32 range: every output is a weighted mean of
    them, so it is finite and, relatively, as near float64 as any other."""
    import torch
    g = torch.Generator().manual_seed(HD)
    T, LMAX = 300, 1024
    q, k = torch.randn((T, NH, HD), generator=g) * 0.1, torch.randn((NKV, LMAX, HD), generator=g)
    v = (torch.rand((NKV, LMAX, HD), generator=g) * 0.5 + 0.5) * big
    for pos in (0, LMAX - T):
        got = run(q.cuda(), k.cuda(), v.cuda(), pos).cpu().double()
        ref = want(q, k, v, pos)
        assert float((got - ref).norm() / ref.norm()) < 2e-6
