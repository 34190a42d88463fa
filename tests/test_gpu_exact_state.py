"""The exact (fp32) state kernel on either side of its slice rule (GPU): calls whose
slices are one value tile wide (few chains) and two, odd and even chunk counts
(the output waves run one chunk behind the chain waves), a ragged last chunk, a
single chunk and packed sequences with an empty one.  Bar: the fp32 parity bar of
the other tests (1e-5)."""

from __future__ import annotations

import pytest
import torch

from oracle import inputs
from oracle import kda_oracle as K
from kda_testutil import TOL, assert_close, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,d", [(1, 1, 1, 64), (1, 64, 3, 128), (2, 129, 2, 64), (1, 250, 33, 128),
                                     (5, 70, 7, 128), (1, 192, 65, 64)])
def test_exact_forward(cuda, B, T, H, d):
    import axiom_amd
    x = inputs.make_inputs(B, T, H, d, d, seed=T + H, dtype="fp32", h0_std=0.1)
    print(f"[exact state] B={B} T={T} H={H} d={d}", flush=True)
    t = {n: to_dev(x[n], torch.float32, cuda) for n in x}
    o, ht = axiom_amd.kda_chunk_fwd(t["q"], t["k"], t["v"], t["g"], t["beta"], initial_state=t["h0"])
    torch.cuda.synchronize()
    o_ref, ht_ref = K.chunk_fwd(x["q"], x["k"], x["v"], x["g"], x["beta"], h0=x["h0"], chunk=64)
    assert_close("o", o, o_ref, TOL["fp32"])
    assert_close("ht", ht, ht_ref, TOL["fp32"])


def test_exact_packed_sequences(cuda):
    import axiom_amd
    lengths = [130, 0, 1, 64, 257]
    cu = inputs.cu_seqlens_from_lengths(lengths)
    x = inputs.make_inputs(1, int(cu[-1]), 2, 128, 128, seed=5, dtype="fp32", h0_std=0.1, n_states=len(lengths))
    t = {n: to_dev(x[n], torch.float32, cuda) for n in x}
    o, ht = axiom_amd.kda_chunk_fwd(t["q"], t["k"], t["v"], t["g"], t["beta"], initial_state=t["h0"],
                                    cu_seqlens=torch.from_numpy(cu).to(cuda))
    for i, (s, e) in enumerate(zip(cu[:-1], cu[1:])):
        one = {n: t[n][:, s:e].contiguous() for n in ("q", "k", "v", "g", "beta")}
        if e > s:
            oi, hi = axiom_amd.kda_chunk_fwd(one["q"], one["k"], one["v"], one["g"], one["beta"],
                                             initial_state=t["h0"][i:i + 1].contiguous())
            assert torch.equal(o[:, s:e], oi) and torch.equal(ht[i:i + 1], hi), i
        else:
            assert torch.equal(ht[i], t["h0"][i])


@pytest.mark.parametrize("T", [64, 128, 192, 300])
def test_many_chains_in_short_segments(cuda, T):
    """512 chains run in segments of one to a few chunks, where a segment ends while fragments would still
    be loaded ahead; a row of the batch by itself runs in one.  The same bits."""
    import axiom_amd
    B, H, d = 16, 32, 128
    g = torch.Generator(device=cuda).manual_seed(T)
    R = lambda *s: torch.randn(*s, device=cuda, generator=g)
    q, k = (torch.nn.functional.normalize(R(B, T, H, d), dim=-1) for _ in range(2))
    ops = [q, k, R(B, T, H, d), -torch.nn.functional.softplus(R(B, T, H, d)), torch.sigmoid(R(B, T, H))]
    h0 = R(B, H, d, d) * 0.1
    o, ht = axiom_amd.kda_chunk_fwd(*ops, initial_state=h0)
    for b in (0, B - 1):
        one, h1 = axiom_amd.kda_chunk_fwd(*(x[b:b + 1] for x in ops), initial_state=h0[b:b + 1])
        assert torch.equal(o[b:b + 1], one) and torch.equal(ht[b:b + 1], h1)
