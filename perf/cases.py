"""What this framework's users have it do, as measurable cases.

Two uses of the library: training attention layers (forward with the
log-sum-exp, then the backward) and an inference engine's prefill and decode
over a KV cache. Each listed case stands for a use named at its entry; draw()
gives more of the same ranges. Sizes are the ones of the benchmark, the
configuration table and the prefill table, and ragged ones between them.
"""
import math

import torch

import mx230_amd as mx
from mx230_amd.autograd import CausalSelfAttention

F64 = torch.float64


def _train(name, B, Hq, Hkv, N, d, causal, bf16):
    return {"name": name, "kind": "train", "B": B, "Hq": Hq, "Hkv": Hkv, "N": N, "d": d, "causal": causal,
            "bf16": bf16}


def _cache(name, n_tok, pos0, Hq, Hkv, d, bf16, paged, split):
    return {"name": name, "kind": "cache", "n_tok": n_tok, "pos0": pos0, "Hq": Hq, "Hkv": Hkv, "d": d, "bf16": bf16,
            "paged": paged, "split": split}


def listed():
    return [
        # the benchmark's training step: one attention layer of a 12-head
        # decoder at 4096 tokens
        _train("train_mha", 4, 12, 12, 4096, 64, True, True),
        # the same with grouped-query heads, 7 query heads to a KV head
        _train("train_gqa", 2, 14, 2, 4096, 64, True, True),
        # 128-wide heads, 8 query heads to a KV head, one sequence
        _train("train_gqa_d128", 1, 32, 4, 2048, 128, True, True),
        # an encoder's (non-causal) layer on short sequences of odd length
        _train("train_ragged", 3, 10, 10, 777, 64, False, True),
        # a long document in one sequence, non-causal
        _train("train_long", 1, 12, 12, 32768, 64, False, True),
        # the single-precision training step of the configuration table
        _train("train_fp32", 4, 12, 12, 1024, 64, True, False),
        # the smallest step: one single-precision head of 256 tokens, where
        # launches and the host count
        _train("train_fp32_one_head", 1, 1, 1, 256, 64, False, False),
        # an engine's first chunk of a long prompt into a paged cache
        _cache("prefill_paged", 4096, 0, 32, 4, 64, True, True, False),
        # a later, partly filled chunk against a single-precision cache
        _cache("prefill_chunk_fp32", 500, 3584, 14, 2, 64, False, False, True),
        # one generated token against a paged cache of 4096
        _cache("decode_paged", 1, 4095, 32, 4, 64, True, True, True),
        # one generated token far into a long context
        _cache("decode_long", 1, 65535, 14, 2, 64, True, False, True),
        # a whole attention block (projections by torch, attention by this
        # library) forward and backward under autograd
        {"name": "block", "kind": "block", "B": 2, "N": 1024, "Hq": 14, "Hkv": 2, "d": 64, "bf16": True},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    u = rng.random()
    if u < 0.55:
        bf16 = rng.random() < 0.65
        d = 128 if bf16 and rng.random() < 0.35 else 64
        Hkv, group = rng.choice((1, 2, 3, 4, 8, 12)), rng.choice((1, 1, 1, 2, 4, 7, 8))
        # the work of a drawn step stays below that of the largest listed one
        most = (4.0e12 if bf16 else 8.0e11) / (14.0 * d * Hkv * group)
        N = min(_spread(rng, 64, 8192), int(math.sqrt(most)))
        B = rng.randint(1, max(1, min(8, int(most / (float(N) * N)))))
        return {"kind": "train", "B": B, "Hq": Hkv * group, "Hkv": Hkv, "N": N, "d": d,
                "causal": rng.random() < 0.6, "bf16": bf16}
    if u < 0.92:
        bf16 = rng.random() < 0.7
        d = 128 if bf16 and rng.random() < 0.3 else 64
        Hkv, group = rng.choice((1, 2, 4, 8)), rng.choice((1, 4, 7, 8))
        one = rng.random() < 0.45
        return {"kind": "cache", "n_tok": 1 if one else _spread(rng, 2, 4096),
                "pos0": _spread(rng, 63, 65535) if one else rng.choice((0, _spread(rng, 16, 16384))),
                "Hq": Hkv * group, "Hkv": Hkv, "d": d, "bf16": bf16, "paged": rng.random() < 0.5,
                "split": one or rng.random() < 0.6}
    Hkv, group = rng.choice((1, 2, 4)), rng.choice((1, 4, 7))
    return {"kind": "block", "B": rng.randint(1, 4), "N": _spread(rng, 128, 2048), "Hq": Hkv * group, "Hkv": Hkv,
            "d": rng.choice((64, 128)), "bf16": True}


BLOCK_ROWS = 16  # rows of a paged cache's block, as in the prefill table


def _dtype(case):
    return torch.bfloat16 if case["bf16"] else torch.float32


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def prepare(case, seed):
    g = _gen(seed)
    dt = _dtype(case)
    st = {"case": case}
    if case["kind"] == "train":
        B, Hq, Hkv, N, d = (case[x] for x in ("B", "Hq", "Hkv", "N", "d"))
        st["q"], st["k"], st["v"] = (_randn(g, (B, h, N, d), dt) for h in (Hq, Hkv, Hkv))
        # gradients reach an attention layer far below the activations' size
        st["do"] = _randn(g, (B, Hq, N, d), dt, 0.02)
    elif case["kind"] == "cache":
        n, pos0, Hq, Hkv, d = (case[x] for x in ("n_tok", "pos0", "Hq", "Hkv", "d"))
        # Q is a view of a fused QKV projection's rows, as an engine has it
        st["qkv"] = _randn(g, (n, (Hq + 2 * Hkv) * d), dt)
        st["q"] = st["qkv"][:, :Hq * d]
        rows = pos0 + n
        if case["paged"]:
            # the pool is half as large again as the sequence, its blocks handed out in any order
            nblk = -(-rows // BLOCK_ROWS)
            pool = nblk + nblk // 2 + 1
            st["table"] = torch.randperm(pool, generator=g, device="cuda")[:nblk].to(torch.int32).contiguous()
            rows = pool * BLOCK_ROWS
        st["k"], st["v"] = (_randn(g, (rows, Hkv * d), dt) for _ in range(2))
        st["out"] = torch.empty((n, Hq * d), dtype=dt, device="cuda")
        if case["split"]:
            need = mx.prefill_workspace_bytes(n, pos0, Hq, Hkv, d, case["bf16"])
            st["ws"] = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    else:
        B, N, Hq, Hkv, d = (case[x] for x in ("B", "N", "Hq", "Hkv", "d"))
        dim = Hq * d
        m = CausalSelfAttention(dim, Hq, Hkv, d).to(device="cuda", dtype=dt)
        with torch.no_grad():
            for p in (m.qkv.weight, m.out.weight):
                p.copy_(_randn(g, tuple(p.shape), dt, 1.0 / math.sqrt(p.shape[1])))
        st["m"] = m
        st["x"] = _randn(g, (B, N, dim), dt).requires_grad_(True)
        st["dy"] = _randn(g, (B, N, dim), dt, 0.02)
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "train":
        o, lse = mx.attention_fwd(st["q"], st["k"], st["v"], case["causal"])
        dq, dk, dv = mx.attention_bwd(st["q"], st["k"], st["v"], o, lse, st["do"], case["causal"])
        return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
    if case["kind"] == "cache":
        a = (case["pos0"], case["Hq"], case["Hkv"], case["d"])
        if case["paged"]:
            mx.run_prefill_paged(st["q"], st["k"], st["v"], st["out"], st["table"], BLOCK_ROWS, *a,
                                 split=case["split"], workspace=st.get("ws"))
        elif case["split"]:
            mx.run_prefill_split(st["q"], st["k"], st["v"], st["out"], *a, workspace=st["ws"])
        else:
            mx.run_prefill(st["q"], st["k"], st["v"], st["out"], *a)
        return {"out": st["out"]}
    m, x = st["m"], st["x"]
    y = m(x)
    dx, dwqkv, dwout = torch.autograd.grad(y, (x, m.qkv.weight, m.out.weight), st["dy"])
    return {"y": y, "dx": dx, "dwqkv": dwqkv, "dwout": dwout}


def _pairs(N, causal):
    return N * (N + 1) / 2.0 if causal else float(N) * N


def work(case):
    es = 2 if case["bf16"] else 4
    Hq, Hkv, d = case["Hq"], case["Hkv"], case["d"]
    if case["kind"] == "train":
        B, N = case["B"], case["N"]
        # q, do read, o, dq written; k, v read, dk, dv written; lse written
        nbytes = B * N * d * es * (4 * Hq + 4 * Hkv) + 4 * B * Hq * N
        return {"bytes": nbytes, "flops": 14.0 * _pairs(N, case["causal"]) * d * B * Hq}
    if case["kind"] == "cache":
        n, pos0 = case["n_tok"], case["pos0"]
        nbytes = es * d * (2 * n * Hq + 2 * (pos0 + n) * Hkv)
        if case["paged"]:
            nbytes += 4 * -(-(pos0 + n) // BLOCK_ROWS)
        return {"bytes": nbytes, "flops": 4.0 * (n * float(pos0) + _pairs(n, True)) * d * Hq}
    B, N = case["B"], case["N"]
    dim, wide = Hq * d, (Hq + 2 * Hkv) * d
    weights = dim * wide + dim * dim
    nbytes = es * (2 * weights + 4 * B * N * dim)
    return {"bytes": nbytes, "flops": 6.0 * B * N * weights + 14.0 * _pairs(N, True) * d * B * Hq}


def tolerance(case):
    # Four times the difference from exact() on the MI355X. "max" is large for
    # bf16 because a causal layer's early rows, and the gradients of the keys
    # they see, are many times the root mean square of the rest.
    if not case["bf16"]:
        return {"rel": 5e-6, "max": 1e-4}
    if case["kind"] == "block":
        return {"rel": 1.8e-2, "max": 4e-1}
    return {"rel": 1e-2, "max": 4e-1 if case["kind"] == "train" else 2e-1}


# -------------------------------------------------------------- in 64 bits --

def _attend(q, k, v, do, causal, pos0=0, rows=1024):
    """One head in 64 bits, the query rows in blocks: (o, lse, dq, dk, dv), the
    gradients None without do. Query row i is at position pos0 + i."""
    q, k, v = q.to(F64), k.to(F64), v.to(F64)
    n, d = q.shape
    scale = 1.0 / math.sqrt(d)
    o, lse = torch.empty_like(q), torch.empty(n, dtype=F64, device=q.device)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for i in range(0, n, rows):
        j = min(n, i + rows)
        m = min(k.shape[0], pos0 + j) if causal else k.shape[0]
        s = (q[i:j] @ k[:m].T) * scale
        if causal:
            at = torch.arange(m, device=q.device)[None, :]
            s.masked_fill_(at > torch.arange(pos0 + i, pos0 + j, device=q.device)[:, None], -math.inf)
        lse[i:j] = torch.logsumexp(s, 1)
        p = s.sub_(lse[i:j, None]).exp_()
        o[i:j] = p @ v[:m]
        if do is not None:
            g = do[i:j].to(F64)
            dv[:m] += p.T @ g
            ds = (g @ v[:m].T).sub_((g * o[i:j]).sum(1, keepdim=True)).mul_(p)
            dq[i:j] = (ds @ k[:m]) * scale
            dk[:m] += (ds.T @ q[i:j]) * scale
    return o, lse, dq, dk, dv


def _attend_all(q, k, v, do, causal):
    """[B, H, N, d] heads through _attend."""
    B, Hq, N, d = q.shape
    Hkv = k.shape[1]
    o, dq = (torch.empty((B, Hq, N, d), dtype=F64, device=q.device) for _ in range(2))
    lse = torch.empty((B, Hq, N), dtype=F64, device=q.device)
    dk, dv = (torch.zeros((B, Hkv, N, d), dtype=F64, device=q.device) for _ in range(2))
    for b in range(B):
        for h in range(Hq):
            c = h // (Hq // Hkv)
            o[b, h], lse[b, h], dq[b, h], x, y = _attend(q[b, h], k[b, c], v[b, c], do[b, h], causal)
            dk[b, c] += x
            dv[b, c] += y
    return o, lse, dq, dk, dv


def exact(case, seed):
    st = prepare(case, seed)
    if case["kind"] == "train":
        o, lse, dq, dk, dv = _attend_all(st["q"], st["k"], st["v"], st["do"], case["causal"])
        return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
    Hq, Hkv, d = case["Hq"], case["Hkv"], case["d"]
    if case["kind"] == "cache":
        n, pos0 = case["n_tok"], case["pos0"]
        at = torch.arange(pos0 + n, device="cuda")
        if case["paged"]:
            at = st["table"].long()[at // BLOCK_ROWS] * BLOCK_ROWS + at % BLOCK_ROWS
        out = torch.empty((n, Hq * d), dtype=F64, device="cuda")
        for h in range(Hq):
            c = h // (Hq // Hkv)
            kc, vc = (st[x][at, c * d:(c + 1) * d] for x in ("k", "v"))
            out[:, h * d:(h + 1) * d] = _attend(st["q"][:, h * d:(h + 1) * d], kc, vc, None, True, pos0)[0]
        return {"out": out}
    B, N = case["B"], case["N"]
    x, dy = st["x"].detach().to(F64).reshape(B * N, -1), st["dy"].to(F64).reshape(B * N, -1)
    wqkv, wout = st["m"].qkv.weight.detach().to(F64), st["m"].out.weight.detach().to(F64)

    def heads(t):  # [B N, H d] -> [B, H, N, d]
        return t.reshape(B, N, -1, d).transpose(1, 2).contiguous()

    def flat(t):
        return t.transpose(1, 2).reshape(B * N, -1)

    q, k, v = (heads(t) for t in (x @ wqkv.T).split([Hq * d, Hkv * d, Hkv * d], dim=1))
    o, _, dq, dk, dv = _attend_all(q, k, v, heads(dy @ wout), True)
    dqkv = torch.cat([flat(dq), flat(dk), flat(dv)], dim=1)
    return {"y": (flat(o) @ wout.T).reshape(B, N, -1), "dx": (dqkv @ wqkv).reshape(B, N, -1),
            "dwqkv": dqkv.T @ x, "dwout": dy.T @ flat(o)}
