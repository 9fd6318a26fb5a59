"""The 16-bit forward of one workgroup per query tile (GPU): grids past those whose
tiles share their keys (256 tiles at any head_dim), so many heads of short rows.
Ragged tiles, grouped-query heads, more and fewer queries than keys, block masks with
rows that see nothing, scales of every sign, large logits, the stored LSE and every
small count of kv tiles -- each against 64 bits, with the bars of the parity tests."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import sparse_triton_kernel as stk
from oracle import streaming_oracle as so

pytestmark = pytest.mark.gpu
DEV = "cuda"
# the row sum is of the 16-bit P, each within half a unit: ln(1 + 2^-11), ln(1 + 2^-8)
LSE_BAR = {torch.float16: 5e-4, torch.bfloat16: 4e-3}


def _check(B, H, H_kv, n_q, n_kv, D, dtype, sink, window, mask=None, bm=64, bn=64, scale=None, q_scale=1.0):
    tiles = B * H * -(-n_q // 128)
    print(f"[case] B{B} H{H}/{H_kv} nq{n_q} nkv{n_kv} D{D} {dtype} S{sink} W{window} scale {scale} ({tiles} tiles)",
          flush=True)
    assert tiles > 256
    gen = torch.Generator().manual_seed(n_q + n_kv + D)
    q = (torch.randn(B, H, n_q, D, generator=gen) * q_scale).to(dtype).to(DEV)
    k, v = (torch.randn(B, H_kv, n_kv, D, generator=gen).to(dtype).to(DEV) for _ in range(2))
    causal = mask is None
    if causal:
        mask = stk.make_streaming_mask(n_q, n_kv, stk.StreamingMaskSpec(sink, window), bm, bn, device=DEV)
    out = stk.block_sparse_attention(q.requires_grad_(True), k, v, mask, softmax_scale=scale, block_m=bm, block_n=bn,
                                     is_causal=causal, sink_size=sink, window_size=window, enable_gqa=H != H_kv)
    lse = out.grad_fn.saved_tensors[4].reshape(B, H, n_q)
    vis = torch.from_numpy(so.effective_mask(mask.cpu().numpy(), n_q, n_kv, bm, bn, causal, sink, window)).to(DEV)
    kx, vx = (t.double().repeat_interleave(H // H_kv, 1) for t in (k, v))
    s = torch.matmul(q.detach().double(), kx.transpose(-1, -2).contiguous())
    s = s.mul_(1 / math.sqrt(D) if scale is None else scale).masked_fill_(~vis, -math.inf)
    ref = torch.matmul(torch.nan_to_num(torch.softmax(s, -1)), vx)
    err = (out.detach().double() - ref).abs()
    assert torch.isfinite(err).all()
    assert (err <= 2e-2 + 1e-2 * ref.abs()).all(), float(err.max())
    seen = vis.any(-1).expand(B, H, n_q)
    want = torch.where(seen, torch.logsumexp(s, -1), torch.zeros((), dtype=torch.float64, device=DEV))
    assert (lse[~seen] == 0).all() and (out.detach()[~seen] == 0).all()
    assert float((lse.double() - want).abs().max()) <= LSE_BAR[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("B,H,H_kv,n_q,n_kv,sink,window", [
    (2, 66, 33, 130, 301, 4, 150),      # ragged q and kv tiles, grouped-query, a chunk behind a cache
    (1, 90, 90, 300, 200, 1, 64),       # more queries than keys: rows that see nothing
    (1, 130, 26, 200, 200, 0, 40),      # no sinks, windows shorter than a tile
    (1, 257, 257, 60, 5, 4, 0),         # sinks alone
])
def test_ragged_streams(B, H, H_kv, n_q, n_kv, sink, window, D, dtype):
    _check(B, H, H_kv, n_q, n_kv, D, dtype, sink, window)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_block_mask_with_rows_that_see_nothing(D, dtype):
    rng = np.random.default_rng(D)
    n_q, n_kv, bm, bn = 200, 260, 32, 16
    m = (rng.random((-(-n_q // bm), -(-n_kv // bn))) < 0.35).astype(np.int32)
    m[2] = 0                                            # rows 64 .. 95
    _check(1, 132, 66, n_q, n_kv, D, dtype, 0, 0, mask=torch.from_numpy(m).to(DEV), bm=bm, bn=bn)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("scale,q_scale", [(0.0, 1.0), (-0.3, 1.0), (None, 12.0)])
def test_scales_and_large_logits(scale, q_scale, D, dtype):
    """Scores up to about 60: the reference max moves on most tiles."""
    _check(1, 130, 130, 250, 250, D, dtype, 4, 150, scale=scale, q_scale=q_scale)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n_kv", [64, 100, 128, 192, 256, 300, 320, 384])
def test_kept_tile_counts(n_kv, D, dtype):
    """One query tile that keeps every kv tile, 1 .. 6 of them, even and odd, the last
    ragged at 100 and 300 keys: both loops are unrolled by two, and head_dim 128's is
    skewed by one tile with a peeled last step."""
    _check(1, 257, 257, 128, n_kv, D, dtype, 4, 4096)
