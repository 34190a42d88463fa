"""Calls of the C ABI whose outputs lie over their inputs: the same bits as with buffers of their own.

The forward and the reverse scan share a launch, the seam's gradients leave the kernel
that reads its inputs, and the conv buffers are updated beside the epilogue; each of
these keeps its earlier order where an output shares memory with an input.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kda_testutil import to_dev
from oracle import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,d,prec", [(9, 16, 64, "bf16"), (2, 3, 128, "fp16"), (9, 16, 64, "fp32")])
def test_dh0_over_h0(cuda, B, H, d, prec):
    from axiom_amd import _lib, kda
    T, dt = 70, dict(bf16=torch.bfloat16, fp16=torch.float16, fp32=torch.float32)[prec]
    x = inputs.make_inputs(B, T, H, d, d, seed=3, dtype="bf16", h0_std=0.05)
    q, k, v, g, beta = (to_dev(x[n], dt, cuda) for n in ("q", "k", "v", "g", "beta"))
    h0 = to_dev(x["h0"], torch.float32, cuda)
    do, dht = torch.randn(B, T, H, d, device=cuda), torch.randn(B, H, d, d, device=cuda)
    want = kda.kda_chunk_bwd(q, k, v, g, beta, do, dht=dht, initial_state=h0)
    outs = [torch.empty_like(t) for t in want[:5]]
    ws = torch.empty(kda._ws_bytes("kda_chunk_bwd_workspace", B, T, H, d, d, 64), dtype=torch.uint8, device=cuda)
    p = [t.data_ptr() for t in (q, k, v, g, beta, h0, do, dht, *outs, h0)]
    rc = _lib.lib().kda_chunk_bwd(kda._stream(q.device), *p, B, T, H, d, d, 64, 1.0, kda._IN_CODES[dt],
                                  _lib.KDA_DTYPE_F32, ws.data_ptr(), ws.numel())
    torch.cuda.synchronize()
    assert rc == 0
    for i, (a, w) in enumerate(zip((*outs, h0), want)):
        assert torch.equal(a, w), i


@pytest.mark.parametrize("T,H,d", [(96, 2, 128), (64, 3, 64)])
def test_seam_gradients_over_their_primals(cuda, T, H, d):
    import axiom_amd
    from axiom_amd import _lib, kda
    x = inputs.make_inputs(1, T, H, d, d, seed=T, dtype="bf16", h0_std=0.05)
    rng = np.random.default_rng(T)
    ops = [to_dev(x[n][0].reshape(T, H * d), torch.bfloat16, cuda) for n in ("q", "k", "v")]
    ops.append(to_dev(np.exp(x["g"][0]).reshape(T, H * d), torch.float32, cuda))
    ops.append(to_dev((x["beta"][0][..., None] + rng.uniform(-.05, .05, (T, H, 32))).reshape(T, H * 32),
                      torch.float32, cuda))
    ops.append(to_dev(x["h0"][0], torch.float32, cuda))
    do = torch.randn(T, H * d, device=cuda)
    dS = torch.randn(H, d, d, device=cuda)
    want = axiom_amd.cc_scan_bwd(*ops, do, dS, chunk=32)
    ws = torch.empty(kda._ws_bytes("kda_cc_scan_bwd_batched_workspace", 1, T, H, d, d, 32), dtype=torch.uint8,
                     device=cuda)
    p = [t.data_ptr() for t in (*ops, do, dS, *ops)]
    rc = _lib.lib().kda_cc_scan_bwd_batched(kda._stream(do.device), *p, 1, T, H, d, d, 16, 32, ws.data_ptr(),
                                            ws.numel())
    torch.cuda.synchronize()
    assert rc == 0
    for i, (a, w) in enumerate(zip(ops, want)):
        assert a.dtype == w.dtype and torch.equal(a, w), i


@pytest.mark.parametrize("T,H,d,skip", [(512, 1, 128, 0), (1024, 2, 128, 64), (256, 3, 64, 0)])
def test_seam_state_gradient_over_beta(cuda, T, H, d, skip):
    """dS_in over part of beta32 (from element ``skip`` on): beta32 is read before the scans write dS_in."""
    import axiom_amd
    from axiom_amd import _lib, kda
    x = inputs.make_inputs(1, T, H, d, d, seed=T, dtype="bf16", h0_std=0.05)
    ops = [to_dev(x[n][0].reshape(T, H * d), torch.bfloat16, cuda) for n in ("q", "k", "v")]
    ops.append(to_dev(np.exp(x["g"][0]).reshape(T, H * d), torch.float32, cuda))
    ops.append(to_dev(np.repeat(x["beta"][0], 32, axis=-1), torch.float32, cuda))
    ops.append(to_dev(x["h0"][0], torch.float32, cuda))
    do, dS = torch.randn(T, H * d, device=cuda), torch.randn(H, d, d, device=cuda)
    want = axiom_amd.cc_scan_bwd(*ops, do, dS, chunk=32)
    outs = [torch.empty_like(t) for t in want[:5]]
    dS_in = ops[4].view(-1)[skip:skip + H * d * d]
    assert dS_in.numel() == H * d * d
    ws = torch.empty(kda._ws_bytes("kda_cc_scan_bwd_batched_workspace", 1, T, H, d, d, 32), dtype=torch.uint8,
                     device=cuda)
    p = [t.data_ptr() for t in (*ops, do, dS, *outs, dS_in)]
    rc = _lib.lib().kda_cc_scan_bwd_batched(kda._stream(do.device), *p, 1, T, H, d, d, 16, 32, ws.data_ptr(),
                                            ws.numel())
    torch.cuda.synchronize()
    assert rc == 0
    for i, (a, w) in enumerate(zip((*outs, dS_in.view(H, d, d)), want)):
        assert torch.equal(a, w), i


@pytest.mark.parametrize("T,over", [(2, 0), (333, 1), (130, 2)])
def test_layer_output_over_a_projection(cuda, T, over):
    from axiom_amd import _lib, kda
    B, H, d, K = 2, 4, 64, 4
    xs = [torch.randn(B, T, H * d, device=cuda).to(torch.bfloat16) for _ in range(4)]
    gb = [(-torch.rand(B, T, H, d, device=cuda)).to(torch.bfloat16), torch.rand(B, T, H, device=cuda).to(torch.bfloat16)]
    w = [torch.randn(K, H * d, device=cuda) * 0.4 for _ in range(3)]
    bufs = [torch.randn(B, K - 1, H * d, device=cuda) for _ in range(3)]
    y, ht, new = kda.kda_layer_fwd(*xs[:3], *gb, xs[3], *w, conv_state=tuple(bufs))
    ws = torch.empty(kda._ws_bytes("kda_layer_fwd_workspace", B, T, H, d, K, _lib.KDA_DTYPE_BF16), dtype=torch.uint8,
                     device=cuda)
    ht2 = torch.empty_like(ht)
    p = [t.data_ptr() for t in (*xs[:3], *gb, xs[3], *w, *bufs, *bufs)]
    rc = _lib.lib().kda_layer_fwd(kda._stream(y.device), *p, None, ht2.data_ptr(), xs[over].data_ptr(), None,
                                  B, T, H, d, K, 1.0, 1e-6, _lib.KDA_DTYPE_BF16, _lib.KDA_DTYPE_BF16,
                                  _lib.KDA_DTYPE_BF16, ws.data_ptr(), ws.numel())
    torch.cuda.synchronize()
    assert rc == 0
    assert torch.equal(xs[over], y) and torch.equal(ht2, ht)
    for a, b in zip(bufs, new):
        assert torch.equal(a, b)


@pytest.mark.parametrize("K,T,over", [(4, 1, 0), (4, 2, 2), (3, 1, 1)])
@pytest.mark.parametrize("B,H,d", [(1, 2, 64), (4, 16, 128)])
def test_layer_output_over_an_incoming_buffer(cuda, K, T, over, B, H, d):
    """A call of fewer than K - 1 tokens reads the old buffers; y lies over one, the new ones are elsewhere."""
    from axiom_amd import _lib, kda
    xs = [torch.randn(B, T, H * d, device=cuda).to(torch.bfloat16) for _ in range(4)]
    gb = [(-torch.rand(B, T, H, d, device=cuda)).to(torch.bfloat16), torch.rand(B, T, H, device=cuda).to(torch.bfloat16)]
    w = [torch.randn(K, H * d, device=cuda) * 0.4 for _ in range(3)]
    bufs = [torch.randn(B, K - 1, H * d, device=cuda) for _ in range(3)]
    y, ht, new = kda.kda_layer_fwd(*xs[:3], *gb, xs[3], *w, conv_state=tuple(bufs))
    ws = torch.empty(kda._ws_bytes("kda_layer_fwd_workspace", B, T, H, d, K, _lib.KDA_DTYPE_BF16), dtype=torch.uint8,
                     device=cuda)
    ht2, new2 = torch.empty_like(ht), [torch.empty_like(b) for b in bufs]
    p = [t.data_ptr() for t in (*xs[:3], *gb, xs[3], *w, *bufs, *new2)]
    rc = _lib.lib().kda_layer_fwd(kda._stream(y.device), *p, None, ht2.data_ptr(), bufs[over].data_ptr(), None,
                                  B, T, H, d, K, 1.0, 1e-6, _lib.KDA_DTYPE_BF16, _lib.KDA_DTYPE_BF16,
                                  _lib.KDA_DTYPE_BF16, ws.data_ptr(), ws.numel())
    torch.cuda.synchronize()
    assert rc == 0
    got = bufs[over].view(torch.bfloat16).view(-1)[:y.numel()].view(y.shape)
    assert torch.equal(got, y) and torch.equal(ht2, ht)
    for a, b in zip(new2, new):
        assert torch.equal(a, b)
