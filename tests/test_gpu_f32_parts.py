"""The fp32 kernels whose products run as bf16 parts: tile edges, and operands
that leave the parts' range.

The reference is float64 on the CPU. Tolerance: the parts keep 24 bits and drop
products below 2^-26 of each term, so an output is within the fp32
rounding of its sums, taken as 64 roundings (2^-24 each) of the largest value.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 64 * 2.0 ** -24


def _ref(q, k, v, causal):
    """float64 O and LSE of [H, N, d] queries over [Hkv, N, d] keys."""
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    g = q.shape[0] // k.shape[0]
    k, v = np.repeat(k, g, 0), np.repeat(v, g, 0)
    with np.errstate(invalid="ignore"):
        s = (q @ k.transpose(0, 2, 1)) / math.sqrt(q.shape[-1])
    if causal:
        s = np.where(np.tril(np.ones(s.shape[-2:], bool)), s, -np.inf)
    m = s.max(-1, keepdims=True)
    p = np.exp(s - m)
    l = p.sum(-1, keepdims=True)
    return (p / l) @ v, (m + np.log(l))[..., 0]


def _fwd(q, k, v, causal):
    import torch
    import mx230_amd as mx
    tq, tk, tv = (torch.from_numpy(x[None]).to("cuda") for x in (q, k, v))
    o, lse = mx.attention_fwd(tq, tk, tv, causal)
    torch.cuda.synchronize()
    return o[0].cpu().numpy(), lse[0].cpu().numpy()


def _close(got, want):
    return np.abs(got - want).max() <= TOL * max(1.0, np.abs(want).max())


# 64- and 128-query work-groups (the second from 512 blocks of 128 queries on), every
# remainder of the 16-, 32-, 64- and 128-row tiles
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,Hkv,N", [(1, 1, 1), (1, 1, 31), (2, 1, 33), (1, 1, 64), (3, 3, 65), (4, 2, 129),
                                     (33, 11, 511), (512, 64, 100), (512, 64, 33), (256, 32, 150)])
def test_forward_edges(H, Hkv, N, causal):
    rng = np.random.default_rng(H * 1000 + N)
    q, k, v = (rng.standard_normal((h, N, 64)).astype(np.float32) for h in (H, Hkv, Hkv))
    o, lse = _fwd(q, k, v, causal)
    ro, rl = _ref(q, k, v, causal)
    assert _close(o, ro) and _close(lse, rl)


@pytest.mark.parametrize("H", [1, 171], ids=["g4", "g8"])
def test_forward_outside_the_parts(H):
    """An infinite key element that gives every score -inf (a key no query
    takes), and a value that is finite in fp32 and rounds to infinity in bf16:
    the results are those of fp32 arithmetic."""
    rng = np.random.default_rng(5)
    N = 300
    q, k, v = (rng.standard_normal((H, N, 64)).astype(np.float32) for _ in range(3))
    q[..., 0] = -np.abs(q[..., 0]) - 0.1
    k[:, 77, 0] = np.inf
    # O is summed before it is divided by the row's sum, so a weight of 1 or more
    # relative to the running max (at least the first 64 keys' max, which is
    # positive) would overflow fp32 itself; this key's scores are negative
    k[:, 200] = 0
    k[:, 200, 0] = 8
    v[0, 200, 3] = 3.4e38
    o, lse = _fwd(q, k, v, False)
    keep = np.arange(N) != 77
    ro, rl = _ref(q, k[:, keep], v[:, keep], False)
    assert np.isfinite(o).all()
    for x in range(64):  # per column: the huge value sets its own column's scale
        assert _close(o[..., x], ro[..., x])
    assert _close(lse, rl)


@pytest.mark.parametrize("H", [2, 171], ids=["g4", "g8"])
def test_forward_first_keys_overflow(H):
    """Finite operands whose scores with the first 64 keys all overflow to -inf:
    O and LSE are those over the other keys."""
    rng = np.random.default_rng(12)
    q, k, v = (rng.standard_normal((H, 300, 64)).astype(np.float32) for _ in range(3))
    q[..., 0] = 1e20
    k[..., 0] = 0
    k[:, :64, 0] = -1e20
    o, lse = _fwd(q, k, v, False)
    ro, rl = _ref(q, k[:, 64:], v[:, 64:], False)
    assert _close(o, ro) and _close(lse, rl)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("n,nh,nkv,pos0", [(300, 2, 2, 0), (70, 28, 2, 2100), (8, 4, 2, 2000)], ids=["whole", "g8", "g4"])
def test_first_keys_overflow(n, nh, nkv, pos0, paged):
    """Finite operands whose scores with the first 64 keys (and with those of a
    later split's first stage) all overflow to -inf: those keys have no weight,
    and the rows that see others are the softmax over these."""
    import torch
    import mx230_amd as mx
    rng = np.random.default_rng(11)
    rows = -(-(pos0 + n) // 16) * 16
    q, k, v = (rng.standard_normal((r, c, 64)).astype(np.float32) for r, c in ((n, nh), (rows, nkv), (rows, nkv)))
    q[..., 0] = 1e20
    k[..., 0] = 0
    gone = np.arange(rows) % 1024 < 64
    k[gone, :, 0] = -1e20
    want = np.full((n, nh, 64), np.nan)
    for h in range(nh):
        for i in range(n):
            at = np.flatnonzero(~gone[:pos0 + i + 1])
            if len(at):
                s = k[at, h * nkv // nh].astype(np.float64) @ q[i, h] / 8
                p = np.exp(s - s.max())
                want[i, h] = (p / p.sum()) @ v[at, h * nkv // nh]
    seen = ~np.isnan(want[:, 0, 0])
    assert seen.sum() >= 8
    table = rng.permutation(rows // 16).astype(np.int32)
    kp, vp = np.empty_like(k), np.empty_like(v)
    for i, b in enumerate(table):
        kp[16 * b:16 * b + 16], vp[16 * b:16 * b + 16] = k[16 * i:16 * i + 16], v[16 * i:16 * i + 16]
    tq, tk, tv = (torch.from_numpy(x.reshape(len(x), -1)).cuda() for x in (q, kp if paged else k, vp if paged else v))
    tt = torch.from_numpy(table).cuda()
    for split in (False, True):
        o = torch.empty(n, nh * 64, device="cuda")
        if paged:
            mx.run_prefill_paged(tq, tk, tv, o, tt, 16, pos0, nh, nkv, split=split)
        elif split:
            mx.run_prefill_split(tq, tk, tv, o, pos0, nh, nkv)
        else:
            mx.run_prefill(tq, tk, tv, o, pos0, nh, nkv)
        assert _close(o.cpu().numpy().reshape(n, nh, 64)[seen], want[seen]), split


def _ref_bwd(q, k, v, do, causal):
    """float64 dQ, dK, dV (one head per KV head)."""
    q, k, v, do = (x.astype(np.float64) for x in (q, k, v, do))
    c = 1 / math.sqrt(q.shape[-1])
    with np.errstate(invalid="ignore"):
        s = (q @ k.transpose(0, 2, 1)) * c
    if causal:
        s = np.where(np.tril(np.ones(s.shape[-2:], bool)), s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    dp = do @ v.transpose(0, 2, 1)
    ds = p * (dp - (p * dp).sum(-1, keepdims=True))
    return (ds @ k) * c, (ds.transpose(0, 2, 1) @ q) * c, p.transpose(0, 2, 1) @ do


def _bwd(q, k, v, do, causal):
    import torch
    import mx230_amd as mx
    tq, tk, tv, td = (torch.from_numpy(x[None]).to("cuda") for x in (q, k, v, do))
    o, lse = mx.attention_fwd(tq, tk, tv, causal)
    grads = mx.attention_bwd(tq, tk, tv, o, lse, td, causal)
    torch.cuda.synchronize()
    return [x[0].cpu().numpy() for x in grads]


# dQ and dK cancel (sum_j dS_ij = 0), so their error is that of dS, whose terms
# |P| (|dP| + |Delta|) are up to the row's |dO| |V| ~ 64 for N(0, 1) inputs
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("N", [2, 31, 64, 65, 130, 257])
def test_backward_edges(N, causal):
    rng = np.random.default_rng(N)
    q, k, v, do = (rng.standard_normal((3, N, 64)).astype(np.float32) for _ in range(4))
    for got, want in zip(_bwd(q, k, v, do, causal), _ref_bwd(q, k, v, do, causal)):
        assert np.abs(got - want).max() <= 64 * TOL


def test_backward_outside_the_parts():
    """A key that no query takes for an infinite element: the other keys'
    gradients are those without it, as in fp32 arithmetic. (dQ holds 0 x inf =
    NaN in the infinite element's column, as the sum over keys does.)"""
    rng = np.random.default_rng(9)
    N = 200
    q, k, v, do = (rng.standard_normal((2, N, 64)).astype(np.float32) for _ in range(4))
    q[..., 0] = -np.abs(q[..., 0]) - 0.1
    k[:, 77, 0] = np.inf
    dq, dk, dv = _bwd(q, k, v, do, False)
    keep = np.arange(N) != 77
    rq, rk, rv = _ref_bwd(q, k[:, keep], v[:, keep], do, False)
    assert np.abs(dq[..., 1:] - rq[..., 1:]).max() <= 64 * TOL
    assert np.abs(dk[:, keep] - rk).max() <= 64 * TOL and np.abs(dv[:, keep] - rv).max() <= 64 * TOL
    assert (dk[:, 77] == 0).all() and (dv[:, 77] == 0).all()


# least: the ranges of 64-query blocks, which a workspace has to hold (0: they take none)
@pytest.mark.parametrize("n,nh,nkv,pos0,least", [(70, 28, 2, 2100, 10), (129, 9, 9, 4000, 19), (256, 32, 4, 1000, 4),
                                                 (1200, 14, 2, 1000, 0)])
def test_chunk_split_over_128_query_blocks(n, nh, nkv, pos0, least):
    """An fp32 chunk whose keys are split over 8-wave work-groups: contiguous and
    paged alike, with the whole workspace and every smaller one that holds the
    ranges of 64-query blocks (none where those take none); less is refused."""
    import torch
    import mx230_amd as mx
    rows = -(-(pos0 + n) // 16) * 16
    rng = np.random.default_rng(n)
    q, k, v = (rng.standard_normal((r, c * 64)).astype(np.float32) for r, c in ((n, nh), (rows, nkv), (rows, nkv)))
    table = rng.permutation(rows // 16).astype(np.int32)
    kp, vp = np.empty_like(k), np.empty_like(v)
    for i, b in enumerate(table):
        kp[16 * b:16 * b + 16], vp[16 * b:16 * b + 16] = k[16 * i:16 * i + 16], v[16 * i:16 * i + 16]
    want = np.empty((n, nh * 64))
    for h in range(nh):
        c = slice(h // (nh // nkv) * 64, (h // (nh // nkv) + 1) * 64)
        s = q[:, h * 64:(h + 1) * 64].astype(np.float64) @ k[:pos0 + n, c].T / 8
        s[np.arange(pos0 + n)[None] > pos0 + np.arange(n)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want[:, h * 64:(h + 1) * 64] = (p / p.sum(1, keepdims=True)) @ v[:pos0 + n, c]
    tq, tk, tv, tkp, tvp, tt = (torch.from_numpy(x).cuda() for x in (q, k, v, kp, vp, table))
    need = mx.prefill_workspace_bytes(n, pos0, nh, nkv, 64, False)
    one = n * nh * 66 * 4
    assert need // one > max(least, 1)
    for size in (need, need - one + 4, least * one if least else 16):
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        a, b = (torch.empty(n, nh * 64, device="cuda") for _ in range(2))
        mx.run_prefill_split(tq, tk, tv, a, pos0, nh, nkv, workspace=ws)
        mx.run_prefill_paged(tq, tkp, tvp, b, tt, 16, pos0, nh, nkv, split=True, workspace=ws)
        assert torch.equal(a, b)
        assert _close(a.cpu().numpy(), want)
    if least:
        ws = torch.empty(least * one - 4, dtype=torch.uint8, device="cuda")
        with pytest.raises(mx.MxfaError, match="WORKSPACE"):
            mx.run_prefill_split(tq, tk, tv, a, pos0, nh, nkv, workspace=ws)
        with pytest.raises(mx.MxfaError, match="WORKSPACE"):
            mx.run_prefill_paged(tq, tkp, tvp, b, tt, 16, pos0, nh, nkv, split=True, workspace=ws)


@pytest.fixture(params=[True, False], ids=["one launch", "two launches"])
def launches(request):
    import mx230_amd as mx
    old = mx.set_bwd_options(one_launch=request.param)
    yield
    mx.set_bwd_options(**old)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("Hkv", [8, 1], ids=["mha", "gqa"])
def test_backward_outside_the_parts_everywhere(launches, Hkv, causal):
    """The rows run again in plain fp32 (a key that no query takes for an infinite
    element), in one launch and two, with a GQA group's shares, and from a given
    Delta: the other keys' gradients are those without it."""
    import torch
    import mx230_amd as mx
    rng = np.random.default_rng(10)
    H, N = 8, 200
    q, do = (rng.standard_normal((H, N, 64)).astype(np.float32) for _ in range(2))
    k, v = (rng.standard_normal((Hkv, N, 64)).astype(np.float32) for _ in range(2))
    q[..., 0] = -np.abs(q[..., 0]) - 0.1
    k[:, 77, 0] = np.inf
    keep = np.arange(N) != 77
    kr, vr = (np.repeat(x, H // Hkv, 0) for x in (k, v))
    full = [np.zeros((H, N, 64)) for _ in range(3)]
    for h in range(H):  # one query row at a time over the keys it sees
        for i in range(N):
            at = np.flatnonzero(keep[:i + 1] if causal else keep)
            kk, vv = kr[h, at].astype(np.float64), vr[h, at].astype(np.float64)
            s = kk @ q[h, i].astype(np.float64) / 8
            p = np.exp(s - s.max())
            p /= p.sum()
            dp = vv @ do[h, i].astype(np.float64)
            ds = p * (dp - p @ dp)
            full[0][h, i] = ds @ kk / 8
            full[1][h, at] += np.outer(ds, q[h, i]) / 8
            full[2][h, at] += np.outer(p, do[h, i])
    rq, rk, rv = full[0], *(x.reshape(Hkv, H // Hkv, N, 64).sum(1) for x in full[1:])
    tq, tk, tv, td = (torch.from_numpy(x[None]).to("cuda") for x in (q, k, v, do))
    assert (mx.bwd_workspace_bytes(tq, tk, causal) > 0) == (Hkv == 1)
    o, lse = mx.attention_fwd(tq, tk, tv, causal)
    given = [torch.empty_like(x) for x in (tq, tk, tv)]
    delta = torch.empty_like(lse)
    mx.run_preprocess(td, o, delta)
    mx.run_bwd_flash(tq, tk, tv, td, lse, delta, *given, causal)
    for got in (mx.attention_bwd(tq, tk, tv, o, lse, td, causal), given):
        dq, dk, dv = (x[0].cpu().numpy() for x in got)
        assert np.abs(dq[..., 1:] - rq[..., 1:]).max() <= 64 * TOL
        # a key of a GQA group sums its heads' terms
        assert np.abs(dk[:, keep] - rk[:, keep]).max() <= 64 * TOL * (H // Hkv)
        assert np.abs(dv[:, keep] - rv[:, keep]).max() <= 64 * TOL * (H // Hkv)
        assert (dk[:, 77] == 0).all() and (dv[:, 77] == 0).all()


@pytest.mark.parametrize("which", ["v", "do"])
def test_small_values_keep_their_bits(launches, which):
    """V or dO times 2^-100: O, dQ and dK (dV with dO) are those of the unscaled
    operand times 2^-100, bit for bit (no normal fp32 value is held in fewer
    bits), but for what cancels to the size of the smallest normals."""
    rng = np.random.default_rng(3)
    x = {n: (rng.uniform(0.5, 1.5, (3, 200, 64)) * rng.choice((-1, 1), (3, 200, 64))).astype(np.float32)
         for n in ("q", "k", "v", "do")}
    y = dict(x)
    y[which] = np.ldexp(x[which], -100)
    for causal in (False, True):
        a, b = ([_fwd(z["q"], z["k"], z["v"], causal)[0], *_bwd(z["q"], z["k"], z["v"], z["do"], causal)] for z in (x, y))
        for i, (got, want) in enumerate(zip(b, a)):
            scaled = i in ((0, 1, 2) if which == "v" else (1, 2, 3))
            want = np.ldexp(want, -100) if scaled else want
            normal = np.abs(want) >= 2.0 ** -118
            assert normal.mean() > 0.98 and np.array_equal(got[normal], want[normal]), (causal, i)
            assert np.abs(got[~normal] - want[~normal]).max(initial=0) <= 2.0 ** -126, (causal, i)


# the relative error (2-norm) is 3e-7 to 5e-7 at every size: 16 roundings of 2^-24
@pytest.mark.parametrize("sizes", [(-118, 118, 0, 0), (118, -118, 0, 0), (-10, 10, -52, -52), (0, 0, -118, 0),
                                   (0, 0, 0, -118)], ids=str)
def test_small_against_large(launches, sizes):
    """Q, K, V and dO of sizes 2^sizes whose scores are ordinary ones."""
    rng = np.random.default_rng(4)
    q, k, v, do = (np.ldexp(rng.standard_normal((2, 200, 64)).astype(np.float32), e) for e in sizes)
    got = [_fwd(q, k, v, True)[0], *_bwd(q, k, v, do, True)]
    for x, want in zip(got, [_ref(q, k, v, True)[0], *_ref_bwd(q, k, v, do, True)]):
        c = np.abs(want).max()
        assert np.linalg.norm((x - want) / c) <= 16 * 2.0 ** -24 * np.linalg.norm(want / c)


@pytest.mark.parametrize("Hkv", [4, 2], ids=["mha", "gqa"])
def test_backward_in_place(launches, Hkv):
    """dQ over O's memory, and dK and dV over K's and V's: the results of
    separate outputs (a call whose outputs share memory with its inputs keeps
    the two launches, between which those are no longer read)."""
    import torch
    import mx230_amd as mx
    torch.manual_seed(8)
    q, do = (torch.randn(2, 4, 300, 64, device="cuda") for _ in range(2))
    k, v = (torch.randn(2, Hkv, 300, 64, device="cuda") for _ in range(2))
    o, lse = mx.attention_fwd(q, k, v, True)
    delta = torch.empty_like(lse)
    old = mx.set_bwd_options(one_launch=False)
    dq, dk, dv = (torch.empty_like(x) for x in (q, k, v))
    mx.run_bwd(q, k, v, o, do, lse, delta, dq, dk, dv, True)
    mx.set_bwd_options(**old)
    o2 = o.clone()
    mx.run_bwd(q, k, v, o2, do, lse, delta, o2, dk2 := torch.empty_like(k), dv2 := torch.empty_like(v), True)
    assert torch.equal(o2, dq) and torch.equal(dk2, dk) and torch.equal(dv2, dv)
    k2, v2, dq2 = k.clone(), v.clone(), torch.empty_like(q)
    mx.run_bwd(q, k2, v2, o, do, lse, delta, dq2, k2, v2, True)
    assert torch.equal(dq2, dq) and torch.equal(k2, dk) and torch.equal(v2, dv)


@pytest.mark.parametrize("Hkv,N,causal", [(4, 1, True), (4, 65, False), (2, 300, True), (1, 513, False)])
@pytest.mark.parametrize("finite", [True, False])
def test_one_launch_equals_two_launches(Hkv, N, causal, finite):
    """The one-launch fp32 backward gives the two launches' bits, also where the
    work-groups run again in plain fp32 (an infinite key element)."""
    import torch
    import mx230_amd as mx
    torch.manual_seed(N)
    q, do = (torch.randn(2, 4, N, 64, device="cuda") for _ in range(2))
    k, v = (torch.randn(2, Hkv, N, 64, device="cuda") for _ in range(2))
    if not finite:
        q[..., 0] = -q[..., 0].abs() - 0.1
        k[:, :, N // 2, 0] = float("inf")
    o, lse = mx.attention_fwd(q, k, v, causal)
    res = []
    for one in (True, False):
        old = mx.set_bwd_options(one_launch=one)
        res.append(mx.attention_bwd(q, k, v, o, lse, do, causal))
        mx.set_bwd_options(**old)
    for a, b in zip(*res):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("pos0", [4095, 65535])
def test_long_context_token(pos0):
    """One token over a long cache split into 32 ranges: the rms error of O, over
    16 draws, stays within 8 roundings of 2^-24 (the scores' about 2.5, the sums
    within a stage as much, adding a range's 32 stages 2, the merge 1; rounding
    O's sum 12 times a stage and the scores at the size of the running maximum
    gave 16)."""
    import torch
    import mx230_amd as mx
    err = size = 0.0
    for seed in range(16):
        g = torch.Generator(device="cuda").manual_seed(seed)
        q = torch.randn(1, 4 * 64, generator=g, device="cuda")
        k, v = (torch.randn(pos0 + 1, 64, generator=g, device="cuda") for _ in range(2))
        o = torch.empty_like(q)
        mx.run_prefill_split(q, k, v, o, pos0, 4, 1)
        s = q.double().view(4, 64) @ k.double().t().contiguous() / 8
        want = (torch.softmax(s, -1) @ v.double()).view(1, -1)
        err += float((o - want).square().sum())
        size += float(want.square().sum())
    assert (err / size) ** 0.5 <= 8 * 2.0 ** -24
