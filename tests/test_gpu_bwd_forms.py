"""The forms of the 16-bit backward (GPU): a scale whose power of two rides in an
operand, one that is multiplied in after, and one that cannot divide the LSE."""

from __future__ import annotations

import math

import pytest
import torch

import sparse_triton_kernel as stk
from oracle import streaming_oracle as so

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gradients64(q, k, v, do, vis, scale, o=None, cast=None):
    """dQ, dK, dV in 64 bits; with ``o`` and ``cast``, the reference's rounding: Delta
    over the stored O, P and the scaled dS cast, results in the storage type."""
    q, k, v, do = (t.detach().double() for t in (q, k, v, do))
    p = torch.nan_to_num_(torch.softmax((q @ k.transpose(-1, -2)).mul_(scale).masked_fill_(~vis, -math.inf), -1))
    delta = (do * (p @ v if o is None else o.double())).sum(-1, keepdim=True)
    ds = p * (do @ v.transpose(-1, -2) - delta) * scale
    if cast is None:
        return ds @ k, ds.transpose(-1, -2) @ q, p.transpose(-1, -2) @ do
    p, ds = p.to(cast).double(), ds.to(cast).double()
    return (ds @ k).to(cast), (ds.transpose(-1, -2) @ q).to(cast), (p.transpose(-1, -2) @ do).to(cast)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("scale", [0.0, -0.3, 0.3, 3.0, 0.25, -0.125, 1 / 128, 1e-3, 1e-12])
def test_every_form_and_head_dim_matches_64_bits(scale, D, dtype):
    """Each scale class at each head dim, on ragged tiles and rows that see nothing
    (more queries than keys): no further from 64 bits than the reference's
    rounding puts them, 2% and 2^-14 left for the order of sums."""
    print(f"[case] scale {scale} D{D} {dtype}", flush=True)
    B, H, n_q, n_kv, S, W = 1, 2, 300, 270, 4, 64
    gen = torch.Generator().manual_seed(D + 1)
    q, k, v, do = (torch.randn(B, H, n, D, generator=gen).to(dtype).to(DEV) for n in (n_q, n_kv, n_kv, n_q))
    mask = stk.make_streaming_mask(n_q, n_kv, stk.StreamingMaskSpec(S, W), 64, 64, device=DEV)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = stk.block_sparse_attention(*leaves, mask, softmax_scale=scale, is_causal=True, sink_size=S, window_size=W)
    out.backward(do)
    vis = torch.from_numpy(so.token_mask(n_q, n_kv, S, W)).to(DEV)
    exact = _gradients64(q, k, v, do, vis, scale)
    model = _gradients64(q, k, v, do, vis, scale, out.detach(), dtype)
    for name, got, want, ref in zip(("dQ", "dK", "dV"), (t.grad for t in leaves), exact, model):
        got, ref = got.double(), ref.double()
        if not want.any():
            assert not got.any(), name
            continue
        err, bar = (float((x - want).norm() / want.norm()) for x in (got, ref))
        print(f"  {name} {err:.3e} (the reference's rounding {bar:.3e})", flush=True)
        assert err <= 1.02 * bar + 2.0**-14, (name, err, bar)


@pytest.mark.parametrize("D,scale", [(32, None), (128, None), (16, 0.2), (64, 0.1)])
@pytest.mark.parametrize("small,size", [("do", 1e-3), ("do", 1e-4), ("do", 1e-5), ("v", 1e-3)])
def test_fp16_small_gradients_keep_the_accuracy_of_the_reference_rounding(D, scale, small, size):
    """Gradients of training without loss scaling sit among the subnormal numbers of
    fp16, where a factor taken out of an operand or of dS costs accuracy. With a
    scale that is no power of two, dQ and dK are no further from 64 bits than the
    reference's rounding (operands as given, dS cast after the scale) puts them;
    10% and the results' own 2^-11 are left for the order of sums."""
    print(f"[case] D{D} scale {scale} {small} {size}", flush=True)
    B, H, N, S, W = 1, 2, 512, 4, 64
    gen = torch.Generator().manual_seed(D)
    q, k, v, do = (torch.randn(B, H, N, D, generator=gen) for _ in range(4))
    if small == "do":
        do *= size
    else:
        v *= size
    q, k, v, do = (t.to(torch.float16).to(DEV) for t in (q, k, v, do))
    mask = stk.make_streaming_mask(N, N, stk.StreamingMaskSpec(S, W), 64, 64, device=DEV)
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = stk.block_sparse_attention(*leaves, mask, softmax_scale=scale, is_causal=True, sink_size=S, window_size=W)
    out.backward(do)
    vis = torch.from_numpy(so.token_mask(N, N, S, W)).to(DEV)
    scale = scale or 1.0 / math.sqrt(D)
    exact = _gradients64(q, k, v, do, vis, scale)
    model = _gradients64(q, k, v, do, vis, scale, out.detach(), torch.float16)
    for name, got, want, ref in zip(("dQ", "dK"), (leaves[0].grad, leaves[1].grad), exact, model):
        err = float((got.double() - want).norm() / want.norm())
        bar = 1.1 * float((ref.double() - want).norm() / want.norm()) + 2.0**-11
        print(f"  {name} {err:.3e} (bar {bar:.3e})", flush=True)
        assert err <= bar, (name, err, bar)
