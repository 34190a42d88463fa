"""The chunked backward at the edges of its 16-row tiles (GPU): lengths on either
side of a tile and of a chunk, with decays that send some diagonal tiles of a
chunk down the per-element path (a tile that decays by more than 2^-32 in a
channel) beside tiles that stay on the matrix cores.

Bars: those of the other backward tests.  fp32 inputs 1e-4 (their products run
as bf16 hi/lo triples, about 2^-16 each); 16-bit inputs 1e-3 / 2e-3 against the
float64 oracle (fp16 forward-side workspace).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import inputs
from oracle import kda_oracle as K
from kda_testutil import TDT, to_dev

pytestmark = pytest.mark.gpu

NAMES = ("dq", "dk", "dv", "dg", "dbeta", "dh0")


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("T,prec", [(1, "fp32"), (15, "bf16"), (16, "fp32"), (17, "bf16"), (33, "fp16"),
                                    (48, "fp32"), (63, "bf16"), (65, "fp32"), (79, "bf16"), (144, "bf16")])
def test_bwd_at_tile_edges_with_mixed_decay(cuda, T, prec, d):
    import axiom_amd
    H = 2
    x = inputs.make_inputs(1, T, H, d, d, seed=T + d, dtype="bf16" if prec != "fp32" else "fp32", h0_std=0.05)
    # every third token of head 1 decays a quarter of the channels by e^-12 more: tiles past 2^-32
    # (six such tokens: 2^-104) beside channels and a head that stay far above it
    x["g"][:, ::3, 1, : d // 4] -= 12.0
    x["g"] = np.asarray(torch.from_numpy(x["g"]).to(TDT[prec]).float())
    rng = np.random.default_rng(T)
    do = rng.standard_normal((1, T, H, d)).astype(np.float32)
    dS = rng.standard_normal((1, H, d, d)).astype(np.float32) * 0.1
    t = {n: to_dev(x[n], TDT[prec], cuda) for n in ("q", "k", "v", "g", "beta")}
    print(f"[bwd tiles] T={T} d={d} {prec}", flush=True)
    got = axiom_amd.kda_chunk_bwd(*(t[n] for n in ("q", "k", "v", "g", "beta")), to_dev(do, torch.float32, cuda),
                                  dht=to_dev(dS, torch.float32, cuda), initial_state=to_dev(x["h0"], torch.float32, cuda))
    torch.cuda.synchronize()
    xs = {n: t[n].double().cpu().numpy() for n in t}
    ref = K.chunk_bwd(*(xs[n] for n in ("q", "k", "v", "g", "beta")), do.astype(np.float64),
                      dht=dS.astype(np.float64), h0=x["h0"], chunk=16)
    rel_tol, abs_tol = (1e-4, 1e-4) if prec == "fp32" else (1e-3, 2e-3)
    for n, a, b in zip(NAMES, got, ref):
        a = a.double().cpu().numpy()
        assert np.all(np.isfinite(a)), n
        rel, mx = K.rel_l2(a, b), K.max_abs(a, b)
        print(f"  {n}: rel_l2={rel:.2e} max_abs={mx:.2e}")
        assert rel <= rel_tol and mx <= abs_tol * max(1.0, float(np.abs(b).max())), n


@pytest.mark.parametrize("B,T", [(31, 64), (32, 64), (32, 37), (32, 65)])
def test_many_one_chunk_chains(cuda, B, T):
    """fp32, d = 64: the forward scan in a launch of its own from 1 024 one-chunk chains on.  A chain's
    gradients do not depend on the others: the same bits as in a call of one batch row."""
    import axiom_amd
    H, d = 32, 64
    x = inputs.make_inputs(B, T, H, d, d, seed=T, dtype="fp32", h0_std=0.1)
    t = {n: to_dev(x[n], torch.float32, cuda) for n in x}
    g = torch.Generator(device=cuda).manual_seed(1)
    do, dht = torch.randn(B, T, H, d, device=cuda, generator=g), torch.randn(B, H, d, d, device=cuda, generator=g)
    ops = [t[n] for n in ("q", "k", "v", "g", "beta")]
    got = axiom_amd.kda_chunk_bwd(*ops, do, dht=dht, initial_state=t["h0"])
    for b in (0, B // 2, B - 1):
        s = slice(b, b + 1)
        one = axiom_amd.kda_chunk_bwd(*(y[s] for y in ops), do[s], dht=dht[s], initial_state=t["h0"][s])
        for i, (u, v) in enumerate(zip(got, one)):
            assert torch.equal(u[s], v), (b, i)
