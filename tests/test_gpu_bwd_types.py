"""Gradients in the primals' 16-bit types and the seam's own operands (GPU): the
kernels that form a gradient round it as a cast of the fp32 result would, bit
for bit, and the cc_scan backward gives the same bits whether its operands'
alignment lets the kernels take them directly or sends them through the
element-wise passes before and after the dense backward."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import inputs
from kda_testutil import TDT, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,d,prec,gates", [(1, 1, 64, "bf16", "same"), (65, 3, 128, "bf16", "same"),
                                              (79, 2, 64, "fp16", "same"), (130, 2, 128, "fp16", "same"),
                                              (47, 2, 128, "bf16", "fp32")])
def test_rounded_gradients_equal_a_cast(cuda, T, H, d, prec, gates):
    import axiom_amd
    from axiom_amd import kda
    x = inputs.make_inputs(2, T, H, d, d, seed=T, dtype="bf16", h0_std=0.05)
    gdt = torch.float32 if gates == "fp32" else TDT[prec]
    q, k, v = (to_dev(x[n], TDT[prec], cuda) for n in ("q", "k", "v"))
    g, beta = (to_dev(x[n], gdt, cuda) for n in ("g", "beta"))
    do = torch.randn(2, T, H, d, device=cuda)
    print(f"[typed gradients] T={T} H={H} d={d} {prec} gates={gates}", flush=True)
    want = axiom_amd.kda_chunk_bwd(q, k, v, g, beta, do)
    got = kda._chunk_bwd(q, k, v, g, beta, do, None, None, 1.0, 64, True, None, q.dtype, g.dtype)
    mixed = kda._chunk_bwd(q, k, v, g, beta, do, None, None, 1.0, 64, True, None, torch.float32, g.dtype)
    torch.cuda.synchronize()
    for i, (a, m, w) in enumerate(zip(got, mixed, want)):
        assert torch.equal(a, w.to(a.dtype)) and torch.equal(m, w.to(m.dtype)), i
    assert mixed[0].dtype == torch.float32 and got[0].dtype == q.dtype and got[3].dtype == g.dtype


@pytest.mark.parametrize("T,d,K", [(1, 64, 1), (37, 128, 4), (70, 64, 8)])
def test_rounded_projection_gradients_equal_a_cast(cuda, T, d, K):
    import axiom_amd
    from axiom_amd import kda
    H = 2
    xs = [torch.randn(2, T, H * d, device=cuda).to(torch.bfloat16) for _ in range(3)]
    ws = [torch.randn(K, H * d, device=cuda) * 0.4 for _ in range(3)]
    dy = [torch.randn(2, T, H, d, device=cuda) for _ in range(3)]
    want, wantw, _ = axiom_amd.kda_prologue_bwd(*xs, *ws, *dy)
    got, gotw, _ = kda._prologue_bwd(*xs, *ws, *dy, None, None, torch.bfloat16)
    torch.cuda.synchronize()
    for a, w in zip(got, want):
        assert a.dtype == torch.bfloat16 and torch.equal(a, w.to(torch.bfloat16))
    for a, w in zip(gotw, wantw):
        assert torch.equal(a, w)


@pytest.mark.parametrize("T,H,d,which", [(96, 2, 128, "alpha"), (64, 3, 64, "beta32"), (160, 1, 128, "alpha")])
def test_seam_backward_of_misaligned_gates_matches(cuda, T, H, d, which):
    import axiom_amd
    x = inputs.make_inputs(1, T, H, d, d, seed=T, dtype="bf16", h0_std=0.05)
    rng = np.random.default_rng(T)
    q, k, v = (to_dev(x[n][0].reshape(T, H * d), torch.bfloat16, cuda) for n in ("q", "k", "v"))
    gates = dict(alpha=to_dev(np.exp(x["g"][0]).reshape(T, H * d), torch.float32, cuda),
                 beta32=to_dev((x["beta"][0][..., None] + rng.uniform(-.05, .05, (T, H, 32))).reshape(T, H * 32),
                               torch.float32, cuda))
    S, do, dS = (to_dev(a.astype(np.float32), torch.float32, cuda) for a in
                 (x["h0"][0], rng.standard_normal((T, H * d)), rng.standard_normal((H, d, d)) * 0.1))
    want = axiom_amd.cc_scan_bwd(q, k, v, gates["alpha"], gates["beta32"], S, do, dS, chunk=32)
    t = gates[which]
    off = torch.empty(t.numel() + 1, device=cuda)[1:].view(t.shape)
    off.copy_(t)
    assert off.data_ptr() % 16 == 4
    gates[which] = off
    got = axiom_amd.cc_scan_bwd(q, k, v, gates["alpha"], gates["beta32"], S, do, dS, chunk=32)
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype and torch.equal(a, b), i


def test_seam_backward_brings_the_dense_workspace_alone(cuda):
    """Beside its outputs a call with aligned gates allocates what the dense backward needs, no room for
    the two-pass form's fp32 gradients and gates (blocks are rounded up to 512 bytes)."""
    import axiom_amd
    from axiom_amd import kda
    T, H, d = 1024, 2, 128
    q, k, v = (torch.randn(T, H * d, device=cuda).to(torch.bfloat16) * 0.1 for _ in range(3))
    alpha, beta32 = torch.rand(T, H * d, device=cuda) * 0.5 + 0.5, torch.rand(T, H * 32, device=cuda)
    S, do, dS = torch.randn(H, d, d, device=cuda), torch.randn(T, H * d, device=cuda), torch.randn(H, d, d, device=cuda)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = axiom_amd.cc_scan_bwd(q, k, v, alpha, beta32, S, do, dS, chunk=32)
    used = torch.cuda.max_memory_allocated() - before
    need = kda._ws_bytes("kda_chunk_bwd_workspace", 1, T, H, d, d, 64) + sum(t.numel() * t.element_size() for t in out)
    assert need <= used <= need + 512 * (len(out) + 1)
