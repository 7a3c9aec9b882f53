"""The prefill of at most 16 query rows per head (the few-row kernels): every
remainder of its 64-key stages and of its waves' turns, split and unsplit,
contiguous and paged, against float64 attention on the CPU.

Tolerance: the result is rounded to bf16 (2^-9 of it) after P was (2^-9 of each
weight), so 2^-7 of the largest value."""
from __future__ import annotations

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [64, 128])
# 1 token: the GQA group's heads are the rows; 16: the most rows of the kernel
@pytest.mark.parametrize("n,nh,nkv,pos0", [
    (1, 1, 1, 0), (1, 7, 1, 62), (1, 7, 1, 63), (1, 16, 1, 64), (1, 8, 2, 511), (1, 8, 2, 512), (1, 4, 4, 1023),
    (1, 14, 2, 1024), (1, 8, 1, 8200), (1, 3, 1, 40000), (16, 2, 1, 100), (16, 2, 1, 1500), (3, 4, 2, 0), (5, 2, 2, 1021),
    # around the ends of the few-row kernels' range: one stage, 192, 256 and more heads,
    # more stages than its waves hold at once
    (1, 144, 144, 1200), (8, 144, 12, 1200), (2, 192, 96, 700), (16, 256, 64, 120), (2, 257, 257, 100), (1, 64, 64, 4100)])
def test_few_rows(n, nh, nkv, pos0, hd):
    import torch
    import mx230_amd as mx
    g = torch.Generator().manual_seed(pos0 + n)
    rows = -(-(pos0 + n) // 16) * 16
    q, k, v = (torch.randn(r, c * hd, generator=g).bfloat16() for r, c in ((n, nh), (rows, nkv), (rows, nkv)))
    table = torch.randperm(rows // 16, generator=g).to(torch.int32)
    kp, vp = (torch.empty_like(x) for x in (k, v))
    for i, b in enumerate(table.tolist()):
        kp[16 * b:16 * b + 16], vp[16 * b:16 * b + 16] = k[16 * i:16 * i + 16], v[16 * i:16 * i + 16]
    q64, k64, v64 = (x.double().numpy() for x in (q, k, v))
    want = np.empty((n, nh * hd))
    for h in range(nh):
        c = slice(h // (nh // nkv) * hd, (h // (nh // nkv) + 1) * hd)
        s = q64[:, h * hd:(h + 1) * hd] @ k64[:pos0 + n, c].T / math.sqrt(hd)
        s[np.arange(pos0 + n)[None] > pos0 + np.arange(n)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want[:, h * hd:(h + 1) * hd] = (p / p.sum(1, keepdims=True)) @ v64[:pos0 + n, c]
    q, k, v, kp, vp, table = (x.cuda() for x in (q, k, v, kp, vp, table))
    out = {}
    for split in (False, True):
        for paged in (False, True):
            o = torch.full((n, nh * hd), float("nan"), dtype=torch.bfloat16, device="cuda")
            if paged:
                mx.run_prefill_paged(q, kp, vp, o, table, 16, pos0, nh, nkv, hd, split=split)
            elif split:
                mx.run_prefill_split(q, k, v, o, pos0, nh, nkv, hd)
            else:
                mx.run_prefill(q, k, v, o, pos0, nh, nkv, hd)
            out[split, paged] = o
            err = np.abs(o.double().cpu().numpy() - want).max()
            assert err <= 2.0 ** -7 * np.abs(want).max(), (split, paged, err)
        assert torch.equal(out[split, False], out[split, True])


def test_workspace_of_32_splits_still_serves():
    """A long context's call takes more than 32 ranges now; a workspace that
    holds 32 (or any number from there) is used for as many."""
    import torch
    import mx230_amd as mx
    pos0, nh, nkv, hd = 20000, 4, 2, 64
    q, k, v = (torch.randn(r, c * hd, device="cuda").bfloat16() for r, c in ((1, nh), (pos0 + 1, nkv), (pos0 + 1, nkv)))
    need = mx.prefill_workspace_bytes(1, pos0, nh, nkv, hd)
    one = nh * (hd + 2) * 4
    assert need > 32 * one
    ref = torch.empty(1, nh * hd, dtype=torch.bfloat16, device="cuda")
    mx.run_prefill(q, k, v, ref, pos0, nh, nkv, hd)
    for size in (32 * one, 50 * one + 16, need):
        o = torch.empty_like(ref)
        mx.run_prefill_split(q, k, v, o, pos0, nh, nkv, hd, workspace=torch.empty(size, dtype=torch.uint8, device="cuda"))
        assert (o.float() - ref.float()).abs().max() <= 2.0 ** -7 * ref.float().abs().max()
    with pytest.raises(mx.MxfaError):
        mx.run_prefill_split(q, k, v, o, pos0, nh, nkv, hd,
                             workspace=torch.empty(32 * one - 16, dtype=torch.uint8, device="cuda"))
