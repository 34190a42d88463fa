"""The calls that a program built on this package makes, at the sizes it makes them.

Every case goes through the public entry points of ``axiom_amd``.  ``listed`` names
the workloads; ``draw`` gives further ones of the same ranges; ``prepare`` makes a
case's inputs on the GPU from a seed; ``run`` is one pass; ``exact`` is the same pass
in 64 bits, written here in plain torch (token recurrence in its chunked WY form,
gradients by autograd through it).

Input distributions are the layer's own: unit-norm q and k rows, standard normal v,
sigmoid betas, log decays ``-softplus(z) e^a`` with one ``a`` in [-2, 0] per head.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import axiom_amd

CHUNK = 64
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # one generated token of one request through the layer: the latency of a single small call
        dict(name="decode_layer_b1", kind="decode_layer", B=1, H=16, d=128, K=4, dtype="bf16"),
        # one decode step of a full serving batch, the state updated in place
        dict(name="decode_b256", kind="decode", B=256, H=16, d=128, dtype="bf16"),
        # a short prompt in full precision: small heads, few chunks
        dict(name="fwd_fp32_t512", kind="fwd", B=1, T=512, H=4, d=64, dtype="fp32", gates="same", h0=False),
        # the next piece of one prompt through the layer, conv history and state carried; a ragged length
        dict(name="layer_prefill_t333", kind="layer_fwd", B=1, T=333, H=16, d=128, K=4, carried=True),
        # the standalone triangular solve with its gradients, as a caller outside the scan uses it
        dict(name="ut_solve_train", kind="ut_train", H=12, C=64, N=256, dtype="fp32"),
        # a batch of sequences, forward only (evaluation, prefill of a batch)
        dict(name="fwd_b4_t4096", kind="fwd", B=4, T=4096, H=16, d=128, dtype="bf16", gates="same", h0=False),
        # one long document: few chains, many chunks
        dict(name="fwd_t65536", kind="fwd", B=1, T=65536, H=16, d=128, dtype="bf16", gates="same", h0=False),
        # packed prompts of very different lengths, each with a state of its own
        dict(name="varlen_64", kind="varlen", N=64, lo=128, hi=8192, lseed=3, H=16, d=128, dtype="bf16"),
        # training steps: the scan alone on a small ragged batch with fp32 gates
        dict(name="chunk_train_d64", kind="chunk_train", B=2, T=1000, H=8, d=64, dtype="bf16", gates="fp32", h0=True),
        # ... in full precision (gradient checks, fp32 training)
        dict(name="chunk_train_fp32", kind="chunk_train", B=2, T=1024, H=8, d=128, dtype="fp32", gates="same", h0=False),
        # ... the reference model's own seam at its geometry (12 heads, 8192 tokens, chunk 32), batched
        dict(name="seam_train_t8192", kind="seam_train", B=2, T=8192, H=12, d=128),
        # ... the layer at the benchmark's shape
        dict(name="layer_train_b4_t4096", kind="layer_train", B=4, T=4096, H=16, d=128, K=4),
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dense(rng, most, t_hi):
    """B, T, H, d with B T H d <= most."""
    d = rng.choice([64, 128, 128])
    H = rng.choice([2, 4, 6, 8, 12, 16, 24, 32])
    B = _spread(rng, 1, 8)
    T = _spread(rng, 17, t_hi)
    T = max(17, min(T, most // (B * H * d)))
    return dict(B=B, T=T, H=H, d=d)


def draw(rng):
    kind = rng.choice(["fwd", "fwd", "varlen", "decode", "decode_layer", "layer_fwd", "chunk_train",
                       "chunk_train", "seam_train", "layer_train", "ut_train"])
    if kind == "fwd":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        gates = rng.choice(["same", "fp32"]) if dtype == "bf16" else "same"
        return dict(kind=kind, **_dense(rng, 1 << 27, 65536), dtype=dtype, gates=gates, h0=rng.random() < 0.5)
    if kind == "varlen":
        lo = _spread(rng, 1, 256)
        return dict(kind=kind, N=_spread(rng, 2, 64), lo=lo, hi=lo + _spread(rng, 64, 6000), lseed=rng.randrange(1000),
                    H=rng.choice([4, 8, 12, 16]), d=rng.choice([64, 128]), dtype=rng.choice(["bf16", "fp16"]))
    if kind == "decode":
        return dict(kind=kind, B=_spread(rng, 1, 256), H=rng.choice([4, 8, 12, 16, 24]), d=rng.choice([64, 128]),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    if kind == "decode_layer":
        return dict(kind=kind, B=_spread(rng, 1, 256), H=rng.choice([4, 8, 12, 16]), d=rng.choice([64, 128]),
                    K=rng.choice([3, 4]), dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind == "layer_fwd":
        return dict(kind=kind, **_dense(rng, 1 << 25, 16384), K=rng.choice([3, 4]), carried=rng.random() < 0.5)
    if kind == "chunk_train":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        gates = rng.choice(["same", "fp32"]) if dtype == "bf16" else "same"
        return dict(kind=kind, **_dense(rng, 1 << 24, 8192), dtype=dtype, gates=gates, h0=rng.random() < 0.5)
    if kind == "seam_train":
        c = _dense(rng, 1 << 25, 8192)
        c["T"] = max(32, c["T"] // 32 * 32)
        return dict(kind=kind, **c)
    if kind == "layer_train":
        return dict(kind=kind, **_dense(rng, 1 << 25, 8192), K=rng.choice([3, 4]))
    return dict(kind=kind, H=_spread(rng, 1, 64), C=rng.choice([16, 32, 48, 64, 64]), N=_spread(rng, 16, 512),
                dtype=rng.choice(["fp32", "fp32", "bf16"]))


# ---------------------------------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _unit(x):
    return x / (x.norm(dim=-1, keepdim=True) + 1e-12)


def _randn(gen, *shape):
    return torch.randn(*shape, device="cuda", generator=gen)


def _log_decay(gen, *shape):
    """-softplus(z) e^a, one a in [-2, 0] per head (the last axis but one)."""
    a = torch.rand(shape[-2], 1, device="cuda", generator=gen) * -2.0
    return -F.softplus(_randn(gen, *shape)) * torch.exp(a)


def _scan_inputs(gen, lead, H, d, dtype, gates="same"):
    dt = DTYPES[dtype]
    gdt = torch.float32 if gates == "fp32" else dt
    q = _unit(_randn(gen, *lead, H, d)).to(dt)
    k = _unit(_randn(gen, *lead, H, d)).to(dt)
    v = _randn(gen, *lead, H, d).to(dt)
    g = _log_decay(gen, *lead, H, d).to(gdt)
    beta = torch.sigmoid(_randn(gen, *lead, H)).to(gdt)
    return dict(q=q, k=k, v=v, g=g, beta=beta)


def _layer_inputs(gen, lead, H, d, K, dtype="bf16"):
    dt = DTYPES[dtype]
    x = {n: _randn(gen, *lead, H * d).to(dt) for n in ("qp", "kp", "vp", "gate")}
    x["g"] = _log_decay(gen, *lead, H, d).to(dt)
    x["beta"] = torch.sigmoid(_randn(gen, *lead, H)).to(dt)
    for n in ("wq", "wk", "wv"):
        x[n] = _randn(gen, K, H * d) * 0.4
    return x


def _lengths(case):
    gen = torch.Generator().manual_seed(case["lseed"])
    return torch.randint(case["lo"], case["hi"] + 1, (case["N"],), generator=gen).tolist()


def _leaves(x, names):
    for n in names:
        x[n] = x[n].detach().requires_grad_(True)
    return x


def _make(case, seed):
    """The inputs of a case, by name (no gradients asked for yet)."""
    gen = _gen(seed)
    kind, H = case["kind"], case["H"]
    if kind == "ut_train":
        C, N, dt = case["C"], case["N"], DTYPES[case["dtype"]]
        low = torch.tril((torch.rand(H, C, C, device="cuda", generator=gen) - 0.5) * 0.5, -1)
        return dict(a=(torch.eye(C, device="cuda") + low).to(dt), b=_randn(gen, H, C, N).to(dt),
                    dx=_randn(gen, H, C, N).to(dt))
    d = case["d"]
    if kind == "varlen":
        cu = [0]
        for n in _lengths(case):
            cu.append(cu[-1] + n)
        x = _scan_inputs(gen, (1, cu[-1]), H, d, case["dtype"])
        x["h0"] = _randn(gen, case["N"], H, d, d) * 0.02
        x["cu"] = torch.tensor(cu, dtype=torch.int32).cuda()
        return x
    B = case["B"]
    if kind == "decode":
        x = _scan_inputs(gen, (B,), H, d, case["dtype"])
        x["S"] = _randn(gen, B, H, d, d) * 0.02
        return x
    if kind in ("decode_layer", "layer_fwd", "layer_train"):
        lead = (B,) if kind == "decode_layer" else (B, case["T"])
        x = _layer_inputs(gen, lead, H, d, case["K"], case.get("dtype", "bf16"))
        if kind == "layer_train":
            x["dy"] = _randn(gen, B, case["T"], H * d).to(torch.bfloat16)
        elif kind == "decode_layer" or case["carried"]:
            for n in ("bq", "bk", "bv"):
                x[n] = _randn(gen, B, case["K"] - 1, H * d)
            x["S"] = _randn(gen, B, H, d, d) * 0.02
        return x
    T = case["T"]
    if kind == "seam_train":
        s = _scan_inputs(gen, (B, T), H, d, "bf16", "fp32")
        x = {n: s[n].reshape(B, T, H * d) for n in ("q", "k", "v")}
        x["alpha"] = torch.exp(s["g"]).reshape(B, T, H * d)
        x["beta32"] = s["beta"].unsqueeze(-1).expand(B, T, H, 32).reshape(B, T, H * 32).contiguous()
        x["S"] = _randn(gen, B, H, d, d) * 0.02
        x["do"] = _randn(gen, B, T, H * d)
        x["dS"] = _randn(gen, B, H, d, d) * 0.1
        return x
    x = _scan_inputs(gen, (B, T), H, d, case["dtype"], case["gates"])
    if case["h0"]:
        x["h0"] = _randn(gen, B, H, d, d) * 0.02
    if kind == "chunk_train":
        x["do"] = _randn(gen, B, T, H, d)
        x["dht"] = _randn(gen, B, H, d, d) * 0.1
    return x


_GRADS = {"ut_train": ("a", "b"), "chunk_train": ("q", "k", "v", "g", "beta"),
          "seam_train": ("q", "k", "v", "alpha", "beta32", "S"),
          "layer_train": ("qp", "kp", "vp", "g", "beta", "gate", "wq", "wk", "wv")}


def _grad_names(case):
    names = _GRADS.get(case["kind"], ())
    return names + ("h0",) if case["kind"] == "chunk_train" and case["h0"] else names


def prepare(case, seed):
    x = _leaves(_make(case, seed), _grad_names(case))
    return dict(case=case, x=x)


# ------------------------------------------------------------------------------------------------ pass

def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "fwd":
        return axiom_amd.kda_chunk_fwd(x["q"], x["k"], x["v"], x["g"], x["beta"], initial_state=x.get("h0"))
    if kind == "varlen":
        return axiom_amd.kda_chunk_fwd(x["q"], x["k"], x["v"], x["g"], x["beta"], initial_state=x["h0"],
                                       cu_seqlens=x["cu"])
    if kind == "decode":
        o = axiom_amd.kda_recurrent_step(x["q"], x["k"], x["v"], x["g"], x["beta"], x["S"])
        return o, x["S"]
    if kind == "decode_layer":
        bufs = (x["bq"], x["bk"], x["bv"])
        y = axiom_amd.kda_decode_layer_step(x["qp"], x["kp"], x["vp"], x["g"], x["beta"], x["gate"],
                                            x["wq"], x["wk"], x["wv"], bufs, x["S"])
        return (y, x["S"]) + bufs
    if kind == "layer_fwd":
        bufs = (x["bq"], x["bk"], x["bv"]) if case["carried"] else None
        y, ht, new = axiom_amd.kda_layer_fwd(x["qp"], x["kp"], x["vp"], x["g"], x["beta"], x["gate"],
                                             x["wq"], x["wk"], x["wv"], conv_state=bufs, initial_state=x.get("S"))
        return (y, ht) + tuple(new)
    leaves = [x[n] for n in _grad_names(case)]
    if kind == "ut_train":
        out = axiom_amd.solve(x["a"], x["b"])
        return (out.detach(),) + torch.autograd.grad(out, leaves, x["dx"])
    if kind == "chunk_train":
        o, ht = axiom_amd.kda_chunk(x["q"], x["k"], x["v"], x["g"], x["beta"], initial_state=x.get("h0"))
        return (o.detach(), ht.detach()) + torch.autograd.grad((o, ht), leaves, (x["do"], x["dht"]))
    if kind == "seam_train":
        o, S = axiom_amd.cc_scan(x["q"], x["k"], x["v"], x["alpha"], x["beta32"], x["S"], tile=16, chunk=32)
        return (o.detach(), S.detach()) + torch.autograd.grad((o, S), leaves, (x["do"], x["dS"]))
    y, ht = axiom_amd.kda_layer(x["qp"], x["kp"], x["vp"], x["g"], x["beta"], x["gate"], x["wq"], x["wk"], x["wv"])
    return (y.detach(), ht.detach()) + torch.autograd.grad(y, leaves, x["dy"])


# ------------------------------------------------------------------------------------------------ work

def work(case):
    """Bytes: every input read once, every output written once.  Operations: the chunked form's products,
    8 C d + 6 d^2 per token and head forward, twice that more for the gradients."""
    kind, H = case["kind"], case["H"]
    if kind == "ut_train":
        C, N, e = case["C"], case["N"], DTYPES[case["dtype"]].itemsize
        # x and dx, dA, dB each once; two solves and the masked outer product
        return dict(bytes=H * (2 * C * C + 4 * C * N) * e, flops=H * 3 * C * C * N)
    d = case["d"]
    tok = 8 * CHUNK * d + 6 * d * d
    st = H * d * d * 4
    if kind in ("decode", "decode_layer"):
        B, e = case["B"], DTYPES[case["dtype"]].itemsize
        if kind == "decode":
            return dict(bytes=B * (2 * st + H * ((4 * d + 1) * e + d * 4)), flops=B * H * 7 * d * d)
        K = case["K"]
        small = H * ((5 * d + 1) * e + d * 4) + 2 * 3 * (K - 1) * H * d * 4
        return dict(bytes=B * (2 * st + small) + 3 * K * H * d * 4, flops=B * H * (7 * d * d + 6 * K * d))
    if kind == "varlen":
        n = sum(_lengths(case)) * H
        e = DTYPES[case["dtype"]].itemsize
        return dict(bytes=n * ((4 * d + 1) * e + d * 4) + 2 * case["N"] * st, flops=n * tok)
    n = case["B"] * case["T"] * H
    if kind in ("layer_fwd", "layer_train"):
        hist = case["B"] * (case["K"] - 1) * H * d * 4 * 3
        bts = n * ((5 * d + 1) * 2 + d * 2) + case["B"] * st + 3 * case["K"] * H * d * 4
        if kind == "layer_fwd":
            return dict(bytes=bts + hist + (hist + case["B"] * st if case["carried"] else 0), flops=n * tok)
        # the backward reads the inputs and dy again and writes a gradient for each input
        return dict(bytes=2 * bts + n * (5 * d + 1) * 2 + 3 * case["K"] * H * d * 4, flops=3 * n * tok)
    if kind == "seam_train":
        ins = n * (3 * d * 2 + d * 4 + 32 * 4) + case["B"] * st
        return dict(bytes=3 * ins + 2 * (n * d * 4 + case["B"] * st), flops=3 * n * tok)
    e = DTYPES[case["dtype"]].itemsize
    eg = 4 if case["gates"] == "fp32" else e
    ins = n * (3 * d * e + (d + 1) * eg) + (case["B"] * st if case["h0"] else 0)
    out = n * d * 4 + case["B"] * st
    if kind == "fwd":
        return dict(bytes=ins + out, flops=n * tok)
    return dict(bytes=3 * ins + 2 * out, flops=3 * n * tok)


def tolerance(case):
    """About four times the distance to the 64-bit results.  16-bit scans run on fp16 operands with fp32 sums;
    gradients and layer outputs are returned in bf16 (half a unit: 2^-9 of each value)."""
    kind = case["kind"]
    if kind in ("decode", "decode_layer"):
        return {"rel": 1e-2, "max": 0.1} if kind == "decode_layer" and case["dtype"] == "bf16" else {"rel": 1e-6, "max": 1e-4}
    if kind in ("fwd", "varlen"):
        return {"rel": 1e-5, "max": 4e-4} if case["dtype"] == "fp32" else {"rel": 2e-3, "max": 4e-2}
    if kind == "chunk_train":
        return {"rel": 2e-5, "max": 1e-3} if case["dtype"] == "fp32" else {"rel": 1e-2, "max": 0.1}
    if kind == "ut_train":
        return {"rel": 2e-6, "max": 1e-4} if case["dtype"] == "fp32" else {"rel": 1e-2, "max": 0.1}
    if kind == "layer_train":      # q, k, v rounded to bf16 between the passes, and the gradients after them
        return {"rel": 2e-2, "max": 0.4}
    return {"rel": 1e-2, "max": 0.2}


# -------------------------------------------------------------------------------------------- 64 bits

def _unit_solve(low, rhs):
    """(I + low)^-1 rhs for strictly lower low [..., C, C], C <= 64: (I - P)(I + P^2)(I + P^4)..., P = low,
    which ends because low^C = 0."""
    x, p = rhs - low @ rhs, low @ low
    for i in range(5):
        x = x + p @ x
        p = p @ p if i < 4 else None
    return x


def _chunked64(q, k, v, g, beta, S):
    """(o [N,T,d], S) for chains q..g [N,T,d], beta [N,T], S [N,d,d], all float64."""
    N, T, d = q.shape
    pad = -T % CHUNK
    if pad:
        q, k, v, g = (F.pad(t, (0, 0, 0, pad)) for t in (q, k, v, g))
        beta = F.pad(beta, (0, pad))
    n = (T + pad) // CHUNK
    q, k, v, g = (t.reshape(N, n, CHUNK, d) for t in (q, k, v, g))
    beta = beta.reshape(N, n, CHUNK, 1)
    G = g.cumsum(2)
    up, down = torch.exp(G), torch.exp(-G)          # a chunk decays by far less than 2^-1000 here
    key = (k * down).transpose(-1, -2).contiguous()
    aqk = torch.tril((q * up) @ key)
    low = torch.tril(beta * ((k * up) @ key), -1)
    W, U = _unit_solve(low, torch.cat([beta * k * up, beta * v], -1)).split(d, -1)
    gq, total = q * up, up[:, :, -1]
    lk = (k * torch.exp(G[:, :, -1:] - G)).transpose(-1, -2).contiguous()
    o = []
    for c in range(n):
        vt = U[:, c] - W[:, c] @ S
        o.append(gq[:, c] @ S + aqk[:, c] @ vt)
        S = total[:, c].unsqueeze(-1) * S + lk[:, c] @ vt
    return torch.cat(o, 1)[:, :T], S


def _scan64(q, k, v, g, beta, S=None):
    """The same for [B,T,H,d] inputs and a [B,H,d,d] state."""
    B, T, H, d = q.shape

    def chains(t):
        return t.transpose(1, 2).reshape(B * H, T, *t.shape[3:])

    S = q.new_zeros(B * H, d, d) if S is None else S.reshape(B * H, d, d)
    o, S = _chunked64(chains(q), chains(k), chains(v), chains(g), chains(beta), S)
    return o.reshape(B, H, T, d).transpose(1, 2), S.reshape(B, H, d, d)


def _conv64(x, w, buf):
    """Causal depthwise conv of x [B,T,C] with taps w [K,C] (w[i] weighs the input i steps back), then swish;
    also the last K - 1 inputs."""
    K, T = w.shape[0], x.shape[1]
    hist = x.new_zeros(x.shape[0], K - 1, x.shape[2]) if buf is None else buf
    full = torch.cat([hist, x], 1)
    a = sum(w[i] * full[:, K - 1 - i:K - 1 - i + T] for i in range(K))
    return a * torch.sigmoid(a), full[:, T:]


def _layer64(x, H, d, one_token=False):
    t = (lambda n: x[n].unsqueeze(1)) if one_token else (lambda n: x[n])
    B, T = t("qp").shape[:2]
    rows, bufs = [], []
    for n in "qkv":
        s, b = _conv64(t(n + "p"), x["w" + n], x.get("b" + n))
        s = s.reshape(B, T, H, d)
        rows.append(s if n == "v" else _unit(s))
        bufs.append(b)
    S = x.get("S")
    o, S = _scan64(*rows, t("g"), t("beta"), S)
    y = torch.sigmoid(t("gate")) * (o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-6)).reshape(B, T, H * d)
    return (y[:, 0] if one_token else y), S, bufs


def exact(case, seed):
    names = _grad_names(case)
    x = {n: t.double() if t.is_floating_point() else t for n, t in _make(case, seed).items()}
    x = _leaves(x, names)
    leaves = [x[n] for n in names]
    kind, H = case["kind"], case["H"]
    if kind == "ut_train":
        out = _unit_solve(torch.tril(x["a"], -1), x["b"])
        return (out.detach(),) + torch.autograd.grad(out, leaves, x["dx"])
    d = case["d"]
    if kind == "fwd":
        return _scan64(x["q"], x["k"], x["v"], x["g"], x["beta"], x.get("h0"))
    if kind == "varlen":
        cu = x["cu"].tolist()
        if cu[-1] * H * d > 1 << 28:
            return None          # minutes of 64-bit work on thousands of chunk positions
        parts = [_scan64(*(x[n][:, s:e] for n in ("q", "k", "v", "g", "beta")), x["h0"][i:i + 1])
                 for i, (s, e) in enumerate(zip(cu, cu[1:]))]
        return torch.cat([p[0] for p in parts], 1), torch.cat([p[1] for p in parts], 0)
    if kind == "decode":
        S = torch.exp(x["g"]).unsqueeze(-1) * x["S"]
        u = (S * x["k"].unsqueeze(-1)).sum(-2)
        S = S + x["k"].unsqueeze(-1) * (x["beta"].unsqueeze(-1) * (x["v"] - u)).unsqueeze(-2)
        return (S * x["q"].unsqueeze(-1)).sum(-2), S
    if kind in ("decode_layer", "layer_fwd"):
        y, S, bufs = _layer64(x, H, d, one_token=kind == "decode_layer")
        return (y, S) + tuple(bufs)
    if kind == "chunk_train":
        o, S = _scan64(x["q"], x["k"], x["v"], x["g"], x["beta"], x.get("h0"))
        return (o.detach(), S.detach()) + torch.autograd.grad((o, S), leaves, (x["do"], x["dht"]))
    if kind == "seam_train":
        B, T = case["B"], case["T"]
        q, k, v, alpha = (x[n].reshape(B, T, H, d) for n in ("q", "k", "v", "alpha"))
        beta = x["beta32"].reshape(B, T, H, 32).mean(-1)
        o, S = _scan64(q, k, v, torch.log(alpha), beta, x["S"])
        o = o.reshape(B, T, H * d)
        return (o.detach(), S.detach()) + torch.autograd.grad((o, S), leaves, (x["do"], x["dS"]))
    y, S, _ = _layer64(x, H, d)
    return (y.detach(), S.detach()) + torch.autograd.grad(y, leaves, x["dy"])
