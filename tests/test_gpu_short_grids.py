"""Forward grids too short for the card (GPU): 16-bit grids of up to 128 128-row
tiles (256 of long lists at head_dim <= 64) share each tile's keys among the waves
of two workgroups, longer ones do not. At the edges -- one kv tile, an odd number of
them, a last half of 64 rows that does not exist, rows that see nothing, both sides
of the lines -- each against the fp64 oracle, with the bars of the parity tests."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import sparse_triton_kernel as stk
from oracle import streaming_oracle as so

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,n_q,n_kv,D,sink,window", [
    (1, 1, 5, 5, 16, 0, 3),             # one tile, a sliver of its rows
    (1, 2, 64, 64, 32, 4, 64),          # the second 64 rows of the tile do not exist
    (1, 2, 65, 129, 64, 1, 200),        # three kv tiles: an odd number, the last of one key
    (1, 1, 130, 700, 128, 4, 40),       # a ragged chunk behind a long cache
    (2, 2, 200, 100, 64, 0, 30),        # more queries than keys: rows that see nothing
    (2, 32, 250, 250, 64, 4, 100),      # 128 tiles
    (1, 64, 250, 250, 128, 4, 100),     # the same, one workgroup per CU
    (2, 64, 250, 250, 64, 4, 100),      # 256 tiles of short lists: one workgroup per tile
    (2, 64, 250, 850, 64, 4, 500),      # 256 of long ones: two
    (2, 64, 250, 850, 16, 4, 500),
    (3, 43, 250, 850, 32, 4, 500),      # 258: one
    (1, 65, 250, 850, 128, 4, 500),     # 130 at head_dim 128: one
    (3, 43, 250, 250, 32, 4, 100),
])
def test_short_grid_matches_oracle(B, H, n_q, n_kv, D, sink, window, dtype):
    print(f"[case] B{B} H{H} nq{n_q} nkv{n_kv} D{D} S{sink} W{window} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(n_q + D)
    q, k, v = (torch.randn(B, H, n, D, generator=gen).to(dtype) for n in (n_q, n_kv, n_kv))
    mask = stk.make_streaming_mask(n_q, n_kv, stk.StreamingMaskSpec(sink, window), 64, 64, device=DEV)
    out = stk.block_sparse_attention(q.to(DEV), k.to(DEV), v.to(DEV), mask, is_causal=True, sink_size=sink,
                                     window_size=window)
    eff = so.effective_mask(mask.cpu().numpy(), n_q, n_kv, 64, 64, True, sink, window)
    ref, _ = so.attention_fwd(*(t.double().numpy() for t in (q, k, v)), eff, 1 / math.sqrt(D))
    err = np.abs(out.double().cpu().numpy() - ref)
    assert np.isfinite(err).all()
    assert (err <= 2e-2 + 1e-2 * np.abs(ref)).all(), err.max()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("B,H,H_kv,n_q,n_kv,sink,window", [
    (2, 4, 4, 130, 130, 4, 50),          # 24 64-row tiles: four workgroups each (dK/dV too, but at D 128)
    (3, 48, 48, 128, 190, 1, 70),        # 288: two each
    (3, 96, 48, 190, 100, 0, 40),        # 864: one each; grouped-query, rows that see nothing
    (1, 48, 48, 700, 700, 4, 100),       # 528 kv columns: the sink column alone is cut
])
def test_fp32_grids_match_oracle(B, H, H_kv, n_q, n_kv, sink, window, D):
    """fp32 forward and backward at each number of workgroups per tile, held to
    1e-5 (N(0, 1) inputs, as the parity tests)."""
    print(f"[case] B{B} H{H}/{H_kv} nq{n_q} nkv{n_kv} D{D} fp32", flush=True)
    gen = torch.Generator().manual_seed(H + D)
    q, do = (torch.randn(B, H, n_q, D, generator=gen) for _ in range(2))
    k, v = (torch.randn(B, H_kv, n_kv, D, generator=gen) for _ in range(2))
    mask = stk.make_streaming_mask(n_q, n_kv, stk.StreamingMaskSpec(sink, window), 64, 64, device=DEV)
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    out = stk.block_sparse_attention(*leaves, mask, is_causal=True, sink_size=sink, window_size=window,
                                     enable_gqa=H != H_kv)
    out.backward(do.to(DEV))
    eff = so.effective_mask(mask.cpu().numpy(), n_q, n_kv, 64, 64, True, sink, window)
    group = H // H_kv
    qn, kn, vn, dn = (t.double().numpy() for t in (q, k, v, do))
    kx, vx = so.expand_kv_heads(kn, group), so.expand_kv_heads(vn, group)
    o, _ = so.attention_fwd(qn, kx, vx, eff, 1 / math.sqrt(D))
    dq, dk, dv = so.attention_bwd(qn, kx, vx, dn, eff, 1 / math.sqrt(D))
    refs = (o, dq, so.reduce_kv_grad(dk, group), so.reduce_kv_grad(dv, group))
    for name, got, ref in zip(("O", "dQ", "dK", "dV"), [out] + [t.grad for t in leaves], refs):
        err = np.abs(got.detach().double().cpu().numpy() - ref)
        assert np.isfinite(err).all() and err.max() <= 1e-5, (name, err.max())
