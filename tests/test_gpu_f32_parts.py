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


# 64- and 128-query work-groups (the second from 129 of 128 queries on), every
# remainder of the 16-, 32-, 64- and 128-row tiles
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,Hkv,N", [(1, 1, 1), (1, 1, 31), (2, 1, 33), (1, 1, 64), (3, 3, 65), (4, 2, 129),
                                     (33, 11, 511), (65, 5, 257)])
def test_forward_edges(H, Hkv, N, causal):
    rng = np.random.default_rng(H * 1000 + N)
    q, k, v = (rng.standard_normal((h, N, 64)).astype(np.float32) for h in (H, Hkv, Hkv))
    o, lse = _fwd(q, k, v, causal)
    ro, rl = _ref(q, k, v, causal)
    assert _close(o, ro) and _close(lse, rl)


@pytest.mark.parametrize("H", [1, 70], ids=["g4", "g8"])
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
